// The decode GEMV's two stages for many batch rows (a prompt through a layer packed for decoding):
// both are products with a sign matrix held as half2-ordered words (element e of a 32-column block
// at bit 15 - e/2 + 16*(e%2)), run as C^T = S X^T on v_mfma_f32_32x32x16.
//
//   stage 1  z[q][j] = s_mid[j] * sum_k sign(V[j,k]) s_in[k] x[q][k], stored as z_hi + z_lo (bf16)
//   stage 2  y[q][i] = sat(s_out[i] * sum_j sign(U[i,j]) (z_hi[q][j] + z_lo[q][j]))
//
// A block takes BP features x BQ batch rows, one wave per 64 features (wave tile 64 x BQ). A word
// shifted left by p carries pair p's signs on bits 15 and 31 of a 16-bit pair; with the word and the
// word shifted by one side by side in 64 bits, one 64-bit shift gives the signs of two pairs, and a
// v_bitop3 each puts them on the s_in pair (stage 1) or on (+1, +1) (stage 2): six VALU per operand of
// 32 features x 16 k, which then feeds BQ / 32 MFMAs (stage 2: as many for z_hi and again for z_lo,
// into the same accumulators).
//
// Every operand reaches LDS by DMA from inline assembly (dma16_lds / dma4_lds), NBUF - 1 steps of 64 k
// ahead; the step barrier waits for the DMAs of the next step only. The x (or z) tile is swizzled at
// fetch time (16-byte chunk p of row r holds the row's chunk p ^ ((r / 2) % 8)), so that operand reads
// have no bank conflicts. A row of words holds only 8 bytes per step, so words are fetched CW words (32
// or 64 contiguous bytes) of a feature at a time: each wave fetches the chunk after the current one for
// its own 64 features, a slice per step, into the third of three chunk buffers. Word pair p of feature
// f lies at p ^ (f / (64 / CW)) % (CW / 2), so that the 32 features one operand reads fall on
// different banks.
//
// A step of 64 k is bound by the latency of its LDS reads and barrier while one block has a CU to itself
// (0.51 us for 512 cycles of MFMAs a wave), and by the matrix cores once the grid is large: stage 2 of
// m = 28672, r = 3520 at 2048 rows runs at 1.46 PFLOP/s (both halves of z counted), stage 1 of the same
// layer at 1.0. The whole op against the kernels it replaced, fp16, us: 11008 x 4096, r = 1632 at 300 / 2048
// rows 53 -> 40, 312 -> 156; 8192 x 28672, r = 3520 at 128 / 666 / 2048 rows 98 -> 56, 1335 -> 220, 3989 ->
// 538.
//
// Small grids: KS groups of waves with buffers of their own share a block's k steps and add their sums
// through LDS; stage 1's k steps may also be split over the grid, the ranges' raw fp32 sums going to
// `part`, which the caller's finishing launch adds in order (deterministic).
#include <algorithm>

#include "nq_gemv_rows.h"

namespace nq {
namespace {

constexpr int NBUF = 3;

__device__ inline uint16_t bf16_of(float v) { return __builtin_bit_cast(uint16_t, static_cast<__bf16>(v)); }
__device__ inline float of_bf16(uint16_t b) { return __uint_as_float(static_cast<uint32_t>(b) << 16); }

// VEC: elements of y per store of stage 2, whose rows are whole pieces of that many (8 or 4; 1 any), apart so that the
// widest does not pay for the others (m = 11008, r = 1632 at 300 rows 22.4 us, 22.55 with the choice in the kernel; m =
// 9804, r = 384 at 579 11.5, 12.0).
template <typename T, typename TO, bool kS2, int BP, int BQ, int CW, int KS, int VEC>
__global__ __launch_bounds__(BP * KS) __attribute__((amdgpu_waves_per_eu(2)))
void rows_kernel(const RowsArgs a, int q_tiles, int p_tiles, int split_steps, int splits) {
    constexpr int NX = kS2 ? 2 : 1;  // x, or z_hi and z_lo
    constexpr int NW = BP / 64;  // waves of a k group
    constexpr int NT = NW * 64;
    constexpr int TP = 2;        // 32-feature tiles of a wave
    constexpr int TQ = BQ / 32;  // 32-row tiles of a wave
    constexpr int KT = 4;        // 16-k tiles of a step
    constexpr int XPT = NX * BQ * 8 / NT;
    constexpr int CWP = CW / 2;             // word pairs (steps) of a chunk
    constexpr int SH = CW == 16 ? 2 : 3;    // features per 64 LDS banks: 1 << SH
    constexpr int RPP = 128 / CW;           // features of the slice fetched in one step
    constexpr int kIssued = XPT + 2 + (kS2 ? 0 : 1);
    static_assert(KS == 1 || KS == 2 || KS == 4, "one, two or four k groups");
    static_assert(CW == 16 || CW == 8, "32 or 64 bytes of a feature per chunk");
    static_assert(NX * BQ * 8 % NT == 0, "the tile's chunks divide evenly");
    __shared__ __attribute__((aligned(16))) uint16_t xsall[KS][NBUF][NX * BQ * 64];
    __shared__ __attribute__((aligned(16))) uint32_t wsall[KS][3][BP * CW];
    __shared__ __attribute__((aligned(16))) uint32_t ssall[KS][NBUF][kS2 ? 4 : NT];
    __shared__ float sos[BP];

    const int grp = KS == 1 ? 0 : __builtin_amdgcn_readfirstlane(threadIdx.x / NT);  // k group
    const int t = static_cast<int>(threadIdx.x) - grp * NT;
    const int lane = t & 63;
    const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
    auto& xs = xsall[grp];
    auto& ws = wsall[grp];
    auto& ss = ssall[grp];
    const int c = lane & 31;
    const int kg = lane >> 5;
    const int tiles = q_tiles * p_tiles;
    const int split = static_cast<int>(blockIdx.x) / tiles;
    const int tile = static_cast<int>(blockIdx.x) - split * tiles;
    const int pt = tile / q_tiles;
    const int q0 = (tile - pt * q_tiles) * BQ;
    const int p0 = pt * BP;
    const int all_steps = a.K / 64;
    // this group's run of the block's k range (of at least KS steps: the host sees to it): the first
    // len % KS groups take one step more, and every group meets the barriers of the longest run
    const int r0 = split * split_steps;
    const int len = min(split_steps, all_steps - r0);
    const int steps = len / KS + (grp < len % KS ? 1 : 0);
    const int first = r0 + grp * (len / KS) + min(grp, len % KS);
    const int run = (len + KS - 1) / KS;

    // DMA sources of the x (z) tile: byte offset of each lane's chunks in their array
    uint32_t xoff[XPT];
    const int ldx = kS2 ? a.zpitch : a.K;
#pragma unroll
    for (int j = 0; j < XPT; ++j) {
        const int ci = (j * NT + t) % (BQ * 8);
        const int r = ci >> 3;
        xoff[j] = 2u * (static_cast<uint32_t>(min(q0 + r, a.batch - 1)) * static_cast<uint32_t>(ldx) +
                        8u * static_cast<uint32_t>((ci & 7) ^ ((r >> 1) & 7)));
    }
    // word slices: lane's dword j of a slice is word position wpos of slice feature wrow[j]
    const int wpos = lane % CW;
    const int wrow0 = lane / CW;  // + 64 / CW for the second dword
    const int f0 = p0 + 64 * wave;
    const uint32_t lx = __builtin_amdgcn_readfirstlane(lds_addr(&xs[0][0]) + static_cast<uint32_t>(wave) * 1024u);
    const uint32_t lw = __builtin_amdgcn_readfirstlane(lds_addr(&ws[0][0]) + static_cast<uint32_t>(wave) * (64u * CW * 4u));
    const uint32_t ls = __builtin_amdgcn_readfirstlane(lds_addr(&ss[0][0]) + static_cast<uint32_t>(wave) * 256u);
    constexpr uint32_t kXBytes = NX * BQ * 128u, kWBytes = BP * CW * 4u, kSBytes = (kS2 ? 4 : NT) * 4u;

    // slice e of chunk ch of this wave's words, into chunk buffer ch % 3
    auto issue_words = [&](int ch, int e) {
        const uint32_t dst = lw + static_cast<uint32_t>(ch % 3) * kWBytes + static_cast<uint32_t>(e) * 512u;
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const int f = RPP * e + j * (64 / CW) + wrow0;  // feature of the wave's 64
            const int pair = (wpos >> 1) ^ ((f >> SH) & (CWP - 1));
            const int word = min(2 * first + ch * CW + 2 * pair + (wpos & 1), a.wpr - 1);
            const uint32_t off = 4u * (static_cast<uint32_t>(min(f0 + f, a.rows - 1)) * static_cast<uint32_t>(a.wpr) +
                                       static_cast<uint32_t>(word));
            dma4_lds(a.words, off, dst + 256u * j);
        }
    };
    // every DMA of step s (clamped to the last one) into step buffer b
    auto issue = [&](int s_, int b) {
        const int s = min(s_, steps - 1);
        const uint32_t k0 = static_cast<uint32_t>(first + s) * 64u;
#pragma unroll
        for (int j = 0; j < XPT; ++j) {
            const uint16_t* src = kS2 ? (j * NT < BQ * 8 ? a.z_hi : a.z_lo) : a.x;
            dma16_lds(src + k0, xoff[j], lx + static_cast<uint32_t>(b) * kXBytes + static_cast<uint32_t>(j * NT * 16));
        }
        if (!kS2) dma4_lds(a.s_in + k0, 4u * static_cast<uint32_t>(lane & 31), ls + static_cast<uint32_t>(b) * kSBytes);
        issue_words(s / CWP + 1, s % CWP);
    };
    static_assert(!kS2 || BQ * 8 % NT == 0, "a DMA round lies in one of the two arrays");

    f32x16 acc[TP][TQ];
#pragma unroll
    for (int tp = 0; tp < TP; ++tp)
#pragma unroll
        for (int tq = 0; tq < TQ; ++tq)
#pragma unroll
            for (int i = 0; i < 16; ++i) acc[tp][tq][i] = 0.0f;
    uint32_t one = T::ONE_PAIR;
    asm volatile("" : "+v"(one));
    const uint32_t mask = 0x80008000u;
    const int xrow = c * 64;

    struct Frag {
        u32x4 s;
        u32x4 x[NX][TQ];
    };
    auto read_kt = [&](Frag& f, const uint16_t* xb, const uint32_t* sb, int kt) {
        const int pos = (2 * kt + kg) ^ ((c >> 1) & 7);
        f.s = kS2 ? u32x4{one, one, one, one} : *reinterpret_cast<const u32x4*>(sb + 8 * kt + 4 * kg);
#pragma unroll
        for (int h = 0; h < NX; ++h)
#pragma unroll
            for (int tq = 0; tq < TQ; ++tq)
                f.x[h][tq] = *reinterpret_cast<const u32x4*>(xb + h * BQ * 64 + xrow + 32 * tq * 64 + 8 * pos);
    };
    // the sign words of a step: w[tp][i] is (word i << 4 kg) and that shifted by one, side by side
    auto read_words = [&](uint2 (&wp)[TP], int s) {
        const uint32_t* wb = &ws[0][0] + static_cast<uint32_t>((s / CWP) % 3) * (BP * CW) + wave * (64 * CW) +
                             c * CW + 2 * ((s % CWP) ^ ((c >> SH) & (CWP - 1)));
#pragma unroll
        for (int tp = 0; tp < TP; ++tp) wp[tp] = *reinterpret_cast<const uint2*>(wb + 32 * tp * CW);
    };
    uint64_t w2[TP][2];
    auto decode_words = [&](const uint2 (&wp)[TP]) {
#pragma unroll
        for (int tp = 0; tp < TP; ++tp) {
            const uint32_t u0 = wp[tp].x << (4 * kg), u1 = wp[tp].y << (4 * kg);
            w2[tp][0] = (static_cast<uint64_t>(u0 << 1) << 32) | u0;
            w2[tp][1] = (static_cast<uint64_t>(u1 << 1) << 32) | u1;
        }
    };
    auto compute_kt = [&](const Frag& g, int kt) {
#pragma unroll
        for (int tp = 0; tp < TP; ++tp) {
            // the bits a shift carries from the low word into the high one land below bit 15
            const uint64_t w01 = w2[tp][kt >> 1] << (8 * (kt & 1));
            const uint64_t w23 = w2[tp][kt >> 1] << (8 * (kt & 1) + 2);
            const u32x4 s = u32x4{g.s.x ^ (static_cast<uint32_t>(w01) & mask),
                                  g.s.y ^ (static_cast<uint32_t>(w01 >> 32) & mask),
                                  g.s.z ^ (static_cast<uint32_t>(w23) & mask),
                                  g.s.w ^ (static_cast<uint32_t>(w23 >> 32) & mask)};
#pragma unroll
            for (int h = 0; h < NX; ++h)
#pragma unroll
                for (int tq = 0; tq < TQ; ++tq) acc[tp][tq] = mfma32x32x16<T>(s, g.x[h][tq], acc[tp][tq]);
        }
    };
    auto sbuf = [&](int b) { return &ss[b][kS2 ? 0 : wave * 64]; };
    Frag f[2];
    uint2 wp[TP];
    // Step s out of buffer b, its first fragments and words already in registers. Once the last k
    // tile's fragments are read the block is done with buffer b: the barrier stands there, before that
    // tile's MFMAs, which then cover the next step's first reads and the issue of step s + NBUF's DMAs.
    auto step = [&](int b, int s) {
        const bool live = KS == 1 || s < steps;  // uniform over the group
        if (live) {
            decode_words(wp);
#pragma unroll
            for (int kt = 0; kt + 1 < KT; ++kt) {
                read_kt(f[(kt + 1) & 1], xs[b], sbuf(b), kt + 1);
                compute_kt(f[kt & 1], kt);
            }
        }
        wait_vmcnt<(NBUF - 2) * kIssued>();  // this wave's DMAs of step s + 1
        barrier_keep_dma();
        read_kt(f[0], xs[(b + 1) % NBUF], sbuf((b + 1) % NBUF), 0);
        read_words(wp, s + 1);
        issue(s + NBUF, b);
        __builtin_amdgcn_sched_barrier(0);
        if (live) compute_kt(f[(KT - 1) & 1], KT - 1);
    };

    for (int e = 0; e < CWP; ++e) issue_words(0, e);
#pragma unroll
    for (int b = 0; b < NBUF; ++b) issue(b, b);
    for (int e = static_cast<int>(threadIdx.x); e < BP; e += NT * KS) {
        const int j = min(p0 + e, a.rows - 1);
        sos[e] = a.scale != nullptr ? TO::to_float(a.scale[j]) : 1.0f;
    }
    wait_vmcnt<(NBUF - 1) * kIssued>();
    barrier_keep_dma();
    read_kt(f[0], xs[0], sbuf(0), 0);
    read_words(wp, 0);
    int s = 0;
    for (; s + NBUF <= run; s += NBUF) {
#pragma unroll
        for (int b = 0; b < NBUF; ++b) step(b, s + b);
    }
#pragma unroll
    for (int b = 0; b + 1 < NBUF; ++b)
        if (s + b < run) step(b, s + b);
    wait_vmcnt<0>();  // the re-fetches of the last steps land before the block's LDS is reused
    __syncthreads();

    // stage 1, K not a multiple of 64: the last K % 64 columns (a multiple of 8), staged through
    // registers with zeros past the row's end
    if (!kS2 && (a.K & 63) != 0 && r0 + len == all_steps) {
        const int k0 = all_steps * 64;
        if (grp == KS - 1) {
            for (int ci = t; ci < BQ * 8; ci += NT) {
                const int r = ci >> 3;
                const int k = k0 + 8 * ((ci & 7) ^ ((r >> 1) & 7));
                u32x4 v = u32x4{0u, 0u, 0u, 0u};
                if (k < a.K)
                    v = *reinterpret_cast<const u32x4*>(a.x + static_cast<size_t>(min(q0 + r, a.batch - 1)) * a.K + k);
                *reinterpret_cast<u32x4*>(&xs[0][ci * 8]) = v;
            }
            if (lane < 32) {
                const int k = k0 + 2 * lane;
                ss[0][kS2 ? 0 : wave * 64 + lane] = k < a.K ? *reinterpret_cast<const uint32_t*>(a.s_in + k) : 0u;
            }
#pragma unroll
            for (int tp = 0; tp < TP; ++tp) {
                const uint32_t* row = a.words + static_cast<size_t>(min(f0 + 32 * tp + c, a.rows - 1)) * a.wpr;
                const int w = all_steps * 2;
                wp[tp] = uint2{row[w], w + 1 < a.wpr ? row[w + 1] : 0u};
            }
        }
        __syncthreads();
        if (grp == KS - 1) {
            decode_words(wp);
#pragma unroll
            for (int kt = 0; kt < KT; ++kt) {
                if (16 * kt < (a.K & 63)) {
                    read_kt(f[0], xs[0], sbuf(0), kt);
                    compute_kt(f[0], kt);
                }
            }
        }
        __syncthreads();
    }

    if constexpr (KS > 1) {  // the other groups' sums join group 0's in order, through the step buffers
        constexpr int kAcc = TP * TQ * 16;
        static_assert(sizeof(xsall) >= (KS - 1) * kAcc * NT * 4, "the step buffers hold the groups' sums");
        float* red = reinterpret_cast<float*>(&xsall[0][0][0]);
        if (grp > 0) {
#pragma unroll
            for (int tp = 0; tp < TP; ++tp)
#pragma unroll
                for (int tq = 0; tq < TQ; ++tq)
#pragma unroll
                    for (int i = 0; i < 16; ++i)
                        red[((grp - 1) * kAcc + (tp * TQ + tq) * 16 + i) * NT + t] = acc[tp][tq][i];
        }
        __syncthreads();
        if (grp == 0) {
#pragma unroll
            for (int g = 0; g < KS - 1; ++g)
#pragma unroll
                for (int tp = 0; tp < TP; ++tp)
#pragma unroll
                    for (int tq = 0; tq < TQ; ++tq)
#pragma unroll
                        for (int i = 0; i < 16; ++i) acc[tp][tq][i] += red[(g * kAcc + (tp * TQ + tq) * 16 + i) * NT + t];
        }
        __syncthreads();
        if (grp > 0) return;
    }

    // acc[tp][tq][4 g4 + e] is feature f0 + 32 tp + 8 g4 + 4 kg + e of batch row q0 + 32 tq + c
    if (!kS2) {
        if (splits > 1) {
            float* plane = a.part + static_cast<size_t>(split) * static_cast<size_t>(a.batch) * a.kpad;
#pragma unroll
            for (int tp = 0; tp < TP; ++tp)
#pragma unroll
                for (int tq = 0; tq < TQ; ++tq)
#pragma unroll
                    for (int g4 = 0; g4 < 4; ++g4) {
                        const int q = q0 + 32 * tq + c;
                        const int j = f0 + 32 * tp + 8 * g4 + 4 * kg;
                        if (q < a.batch && j < a.kpad)
                            *reinterpret_cast<f32x4*>(plane + static_cast<size_t>(q) * a.kpad + j) =
                                f32x4{acc[tp][tq][4 * g4], acc[tp][tq][4 * g4 + 1], acc[tp][tq][4 * g4 + 2],
                                      acc[tp][tq][4 * g4 + 3]};
                    }
            return;
        }
#pragma unroll
        for (int tp = 0; tp < TP; ++tp)
#pragma unroll
            for (int tq = 0; tq < TQ; ++tq)
#pragma unroll
                for (int g4 = 0; g4 < 4; ++g4) {
                    const int q = q0 + 32 * tq + c;
                    const int o = 64 * wave + 32 * tp + 8 * g4 + 4 * kg;
                    const int j = p0 + o;
                    uint16_t hi[4], lo[4];
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        const float v = j + e < a.rows ? acc[tp][tq][4 * g4 + e] * sos[o + e] : 0.0f;
                        hi[e] = bf16_of(v);
                        lo[e] = bf16_of(v - of_bf16(hi[e]));
                    }
                    if (q < a.batch && j < a.kpad) {
                        const size_t at = static_cast<size_t>(q) * a.zpitch + j;
                        *reinterpret_cast<uint2*>(a.z_hi + at) =
                            uint2{hi[0] | (uint32_t(hi[1]) << 16), hi[2] | (uint32_t(hi[3]) << 16)};
                        *reinterpret_cast<uint2*>(a.z_lo + at) =
                            uint2{lo[0] | (uint32_t(lo[1]) << 16), lo[2] | (uint32_t(lo[3]) << 16)};
                    }
                }
        // the columns past kpad that stage 2 reads, in 16-byte pieces (kpad % 32 == 0, zpitch % 64 == 0), shared by the
        // blocks of the batch rows (r = 544, which has 224 such columns, n = 1472, 513 rows: 15.0 us, 26.8 with 2-byte
        // stores of the first block alone)
        const int pieces = (a.zpitch - a.kpad) / 8;
        for (int e = pt * NT + t; e < pieces * BQ; e += p_tiles * NT) {
            const int q = e / pieces;
            if (q0 + q < a.batch) {
                const size_t at = static_cast<size_t>(q0 + q) * a.zpitch + a.kpad + 8 * (e - q * pieces);
                *reinterpret_cast<u32x4*>(a.z_hi + at) = u32x4{0u, 0u, 0u, 0u};
                *reinterpret_cast<u32x4*>(a.z_lo + at) = u32x4{0u, 0u, 0u, 0u};
            }
        }
        return;
    }
    // stage 2: each wave scales and saturates its tile 32 batch rows at a time into 4 KB of the step
    // buffers (64 features of a row are 128 bytes; 16-byte chunk ch of row r at ch ^ ((r / 2) % 8)) and
    // stores whole 128-byte row pieces
    static_assert(sizeof(xsall) >= NW * 4096, "the step buffers hold every wave's piece");
    uint32_t* tb = reinterpret_cast<uint32_t*>(&xsall[0][0][0]) + wave * 1024;
#pragma unroll
    for (int tq = 0; tq < TQ; ++tq) {
#pragma unroll
        for (int tp = 0; tp < TP; ++tp)
#pragma unroll
            for (int g4 = 0; g4 < 4; ++g4) {
                const int o = 64 * wave + 32 * tp + 8 * g4 + 4 * kg;
                uint16_t h[4];
#pragma unroll
                for (int e = 0; e < 4; ++e) h[e] = saturate_to<TO>(acc[tp][tq][4 * g4 + e] * sos[o + e], TO::SAT);
                *reinterpret_cast<uint2*>(tb + 32 * c + 4 * ((4 * tp + g4) ^ ((c >> 1) & 7)) + 2 * kg) =
                    uint2{h[0] | (uint32_t(h[1]) << 16), h[2] | (uint32_t(h[3]) << 16)};
            }
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int rr = (lane >> 3) + 8 * j;
            const u32x4 d = *reinterpret_cast<const u32x4*>(tb + 32 * rr + 4 * ((lane & 7) ^ ((rr >> 1) & 7)));
            const int q = q0 + 32 * tq + rr;
            const int o = f0 + 8 * (lane & 7);
            if (q < a.batch && o < a.rows) {
                uint16_t* dst = a.y + static_cast<size_t>(q) * a.rows + o;
                if constexpr (VEC == 8) {
                    *reinterpret_cast<u32x4*>(dst) = d;
                } else if constexpr (VEC == 4) {
                    *reinterpret_cast<uint2*>(dst) = uint2{d.x, d.y};
                    if (o + 4 < a.rows) *reinterpret_cast<uint2*>(dst + 4) = uint2{d.z, d.w};
                } else {
                    const uint32_t w[4] = {d.x, d.y, d.z, d.w};
#pragma unroll
                    for (int e = 0; e < 8; ++e)
                        if (o + e < a.rows) dst[e] = static_cast<uint16_t>(w[e >> 1] >> (16 * (e & 1)));
                }
            }
        }
    }
}

template <typename T, typename TO, bool kS2, int BP, int BQ, int CW, int KS, int VEC>
void launch_tile(const RowsArgs& a, const RowsPlan& p, hipStream_t st) {
    const int q_tiles = static_cast<int>(ceil_div(a.batch, BQ));
    const int p_tiles = static_cast<int>(ceil_div(a.rows, BP));
    rows_kernel<T, TO, kS2, BP, BQ, CW, KS, VEC><<<dim3(static_cast<unsigned>(q_tiles * p_tiles * p.splits)), BP * KS, 0, st>>>(
        a, q_tiles, p_tiles, p.split_steps, p.splits);
}

// Stage 1 runs these kernels on rows of 512 words or more from 33 batch rows, of 256-511 words from 64,
// on narrower rows from 129; below, the k-split and the 16-row MFMA kernels of nq_gemv.hip are as fast
// or faster (stage 1, fp16, us, those against these: n = 28672, r = 3520 at 32 / 48 / 64 / 128 rows 21.0 /
// 22.3, 32.0 / 24.4, 36.4 / 25.7, 79.2 / 38.1; n = 11008, r = 1632 at 32 / 48 / 64 / 128 rows 11.4 / 12.6,
// 13.5 / 13.5, 15.4 / 14.5, 23.2 / 18.3; n = 4096, r = 1632 at 64 / 96 / 128 rows 8.8 / 11.2, 13.1 / 12.0,
// 13.2 / 13.4).
constexpr int64_t kWideWords = 512, kWideBatch = 33;
constexpr int64_t kMidWords = 256, kMidBatch = 64;
constexpr int64_t kNarrowBatch = 129;
// On rows of up to 256 words the MFMA kernel also stays while its grid is one round of blocks (of 64
// features x 16 batch rows as long as 64 rows of words fit its LDS, of 32 beyond), its time then being that of
// one block (n = 4096, r = 1120 at 200 rows 13.2 against 13.9; at 300 rows, two rounds, 25.0 against 15.5; n =
// 4224, r = 1536 at 129 rows 11.7 / 15.5; n = 8192, r = 512 at 200 / 300 rows 12.7 / 13.3, 24.3 / 15.7), and on
// somewhat longer ones where n % 64 columns would be a tail here (n = 8432, r = 768 at 140 rows 13.0 / 17.1; n =
// 11560, r = 800 at 78 12.8 / 16.6; without a tail 14 / 12 on average there).
constexpr int64_t kMfmaWords64 = 204, kMfmaRoundWords = 256, kMfmaTailWords = 376, kMfmaRoundBlocks = 256;
constexpr int64_t kMinColumns = 512;               // shorter rows are not worth a pipeline
constexpr int64_t kMaxSplits = 16, kMinSteps = 5;  // k ranges, and 64-k steps of the shortest

}  // namespace

// Tile and k ranges with the least estimated time (us). Per 64-k step of a block's longest group, with one
// block on a CU and for each block where several share it: 256 x 64 0.47 / 0.43, 128 x 64 over two k groups
// 0.60 / 0.48, over four 1.05. A launch adds 4 us of start and drain; k ranges add their finishing
// launch (2.5 us) and their sums, written and read at 4.5 TB/s, and run only where they save an eighth of
// the time: they take workspace. (Measured on n = 4096-28672, r = 512-3520 at 96-2048 rows with every tile and
// 1, 2, 3, 4 or 6 ranges. r = 1632, n = 4096 at 300 rows: 256 x 64 33.3 us whole, 18.6 over four ranges, two
// groups 26.0 whole, 16.7 over three, four groups 23.5 whole; n = 28672, r = 3520 at 630 rows: 194 /
// 156 / 193 whole, 180 over two / 224. Blocks of 256 x 128 with waves of 64 x 128, and 128 x 64 in one
// group, were slower but for single cells.)
bool rows_stage1_plan(int64_t batch, int64_t n, int64_t r, int64_t kpad, size_t part_room, RowsPlan& p) {
    const int64_t words = ceil_div(n, 32);
    const int64_t from = words >= kWideWords ? kWideBatch : (words >= kMidWords ? kMidBatch : kNarrowBatch);
    if (batch < from || n % 8 || n < kMinColumns || r <= 0) return false;
    const bool mfma_round = ceil_div(r, words <= kMfmaWords64 ? 64 : 32) * ceil_div(batch, 16) <= kMfmaRoundBlocks;
    if (mfma_round && ((words <= kMfmaRoundWords && batch >= kNarrowBatch) || (words <= kMfmaTailWords && n % 64 != 0)))
        return false;
    const int64_t steps = n / 64;
    struct Shape {
        RowsTile tile;
        int features, groups;
        double alone, shared;  // us a step
    };
    constexpr Shape kShapes[] = {{kRows256, 256, 1, 0.47, 0.43}, {kRows128x2, 128, 2, 0.60, 0.48},
                                 {kRows128x4, 128, 4, 1.05, 1.05}};
    double best = -1.0;
    for (const Shape& s : kShapes) {
        const int64_t tiles = ceil_div(r, s.features) * ceil_div(batch, 64);
        for (int64_t want = 1; want <= kMaxSplits; ++want) {
            const int64_t run = ceil_div(steps, want);
            const int64_t splits = ceil_div(steps, run);  // every range non-empty
            const int64_t last = steps - (splits - 1) * run;
            const size_t bytes = splits > 1 ? static_cast<size_t>(splits) * batch * kpad * 4 : 0;
            if (bytes > part_room || (want > 1 && run < kMinSteps)) break;
            if (last < s.groups) continue;  // every group of the last range has a step
            const int64_t per_cu = ceil_div(tiles * splits, 256);
            double cost = 4.0 + ceil_div(run, s.groups) * (per_cu == 1 ? s.alone : s.shared * per_cu);
            if (splits > 1) cost = 1.15 * (cost + 2.5 + 2.0 * bytes / 4.5e6);
            if (best < 0 || cost < best) {
                best = cost;
                p = RowsPlan{s.tile, static_cast<int>(splits), static_cast<int>(run), bytes};
            }
        }
    }
    return best >= 0;
}

// Stage 2 pays for z_hi and z_lo with two MFMAs per operand, and one block per CU takes 0.74 us a step
// (about as much for each further block of a CU); the kernels that pass over U for 8-32 batch rows at a
// time take time with the batch, about 0.2 us per 1e6 words x rows below 8192 features and 0.135 from
// there on. The less estimated time runs. Measured, us, those against this one: m = 4096, r = 1632 at
// 300 / 666 / 2048 rows 14.3 / 19.6, 29.6 / 22.2, 84 / 43; m = 11008, r = 1632 at 160 / 300 / 2048
// 15.0 / 20.5, 26.5 / 22.5, 157 / 115; m = 28672, r = 3520 at 128 / 300 / 2048 55.7 / 43.3, 137 / 113,
// 792 / 567; m = 1024, r = 512 at 666 / 2048 5.4 / 8.9, 10.7 / 9.2.
//
// A block of 32 batch rows takes a little more than half a step (each decoded sign feeds half the MFMAs) and
// runs where its finer grid leaves the busiest CU less to do. The op, bf16, us, before and with it: m = 8192,
// n = 8192, r = 2240 at 256 / 666 rows 46.6 / 41.3, 90.5 / 89.4; m = 28672, n = 8192, r = 3520 at 64 / 400 rows 51 / 45,
// 197 / 183; m = n = 4096, r = 1120 at 400 / 512 rows 31.6 / 28.3, 34.0 / 29.9; m = n = 2048, r = 1024 at 666 rows
// 35.4 / 27.3. Counted as 0.42 a step it also ran on m = 28672 at 512 rows, 201 / 206; with the other tile's start of
// 2 us also on m = 15153, r = 512 at 94 rows, 14.3 / 15.1.
//
// Short ranks do not hide a block's start behind its steps: up to 28 steps the 64-row block costs 4.8 us and 0.64 a
// step. Counted by the long ranks' figures alone it ran where the passes are faster (stage 2, bf16, us, passes against
// this one: m = 9728, r = 256 at 200 rows 5.5 / 6.8, m = 20480, r = 576 / 1120 at 128 rows 8.4 / 10.3, 14.1 / 16.0, m =
// 12288, r = 640 at 200 rows 10.3 / 11.2; it stays on m = 28672, r = 512 at 128 rows, 11.9 / 10.2).
constexpr double kStart = 2.0, kStep = 0.74, kShortStart = 4.8, kShortStep = 0.64;
constexpr double kHalfStart = 3.5, kHalfStep = 0.43;
bool rows_stage2_plan(int64_t batch, int64_t m, int64_t wr, RowsPlan& p) {
    if (batch < kMidBatch) return false;
    const int64_t steps = ceil_div(wr, 2);
    const int64_t per_cu = ceil_div(ceil_div(m, 256) * ceil_div(batch, 64), 256);
    const int64_t per_cu32 = ceil_div(ceil_div(m, 256) * ceil_div(batch, 32), 256);
    const double rows64 = std::max(kStart + kStep * per_cu * steps, kShortStart + kShortStep * per_cu * steps);
    const double rows32 = kHalfStart + kHalfStep * per_cu32 * steps;
    const bool half = rows32 < rows64;
    const double rows = half ? rows32 : rows64;
    const double passes = 3.0 + 1e-6 * batch * m * wr * (m < 8192 ? 0.2 : 0.135);
    if (rows > passes) return false;
    p = RowsPlan{half ? kRows256q32 : kRows256, 1, static_cast<int>(steps), 0};
    return true;
}

template <typename T>
static void launch_stage1_tile(const RowsArgs& a, const RowsPlan& p, hipStream_t st) {
    if (p.tile == kRows256) launch_tile<T, T, false, 256, 64, 16, 1, 8>(a, p, st);
    else if (p.tile == kRows128x2) launch_tile<T, T, false, 128, 64, 8, 2, 8>(a, p, st);
    else launch_tile<T, T, false, 128, 64, 8, 4, 8>(a, p, st);  // kRows128x4
}

void launch_rows_stage1(int dtype, const RowsArgs& a, const RowsPlan& p, hipStream_t st) {
    if (dtype == NQ_F16) launch_stage1_tile<F16>(a, p, st);
    else launch_stage1_tile<BF16>(a, p, st);
}

template <typename TO, int VEC>
static void launch_stage2_vec(const RowsArgs& a, const RowsPlan& p, hipStream_t st) {
    if (p.tile == kRows256q32) launch_tile<BF16, TO, true, 256, 32, 8, 1, VEC>(a, p, st);
    else launch_tile<BF16, TO, true, 256, 64, 8, 1, VEC>(a, p, st);
}

// 8-byte stores: m = 9804, r = 384 at 579 rows 11.5 us, 21.0 in 2-byte ones.
template <typename TO>
static void launch_stage2_tile(const RowsArgs& a, const RowsPlan& p, hipStream_t st) {
    if (a.rows % 8 == 0 && aligned(a.y, 16)) launch_stage2_vec<TO, 8>(a, p, st);
    else if (a.rows % 4 == 0 && aligned(a.y, 8)) launch_stage2_vec<TO, 4>(a, p, st);
    else launch_stage2_vec<TO, 1>(a, p, st);
}

void launch_rows_stage2(int dtype, const RowsArgs& a, const RowsPlan& p, hipStream_t st) {
    if (dtype == NQ_F16) launch_stage2_tile<F16>(a, p, st);
    else launch_stage2_tile<BF16>(a, p, st);
}

}  // namespace nq
