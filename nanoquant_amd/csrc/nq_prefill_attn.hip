// Attention of a prompt (several tokens per sequence) on a static KV cache: the rotary embedding, the
// cache write and causal attention, as two launches.
//
// 1. kv_rows_kernel rotates the tokens' keys and writes them and the values into the cache rows of
//    their positions.
// 2. prefill_attn_kernel, one block per (sequence, kv head, 128 query rows): the queries of a kv head
//    are rows R = t * G + g (token t, query head g of the group), so grouped heads share the keys and
//    values that a block stages. Each of the four waves keeps 32 rows in registers, rotated as they are
//    loaded, and walks over the cache in tiles of 64 positions with an online softmax:
//      S^T = K Q^T      v_mfma_f32_32x32x16, A = 32 keys x 16 dimensions, B = the wave's queries
//      P^T = exp2(S^T - max), rounded to T for the product (as the torch path rounds its probabilities)
//      O^T += V^T P^T   A = 32 dimensions x 16 keys, B = P^T
//    With S^T rather than S, a lane holds its query's scores, so the row statistics are per lane plus one
//    exchange with lane ^ 32, and P^T's accumulator layout is already a B operand: lane group kg holds
//    keys 4 kg .. +3 and 8 + 4 kg .. +3 of each 16, the key order in which V^T is laid out in LDS. Scores
//    and sums stay in fp32 (the torch path rounds the scores to T).
// 3. A few tokens on a long cache share their keys over the grid in 2, and attn_join_kernel adds the shares.
//
// The scores never reach memory: at 2048 tokens and 32 heads the torch path writes and reads them (256 MB
// in T, 512 MB in fp32) eight times over. What bounds this kernel is issue: per tile and wave 32 MFMAs
// (1024 cycles) and 1500 cycles of VALU (32 exponentials take a third) in 5100 measured ones, a quarter of
// them waits; a SIMD's two waves overlap while both have keys left. Reading operands four ahead of the MFMAs,
// rescaling only when the maximum has grown by kSlack and loads through a uniform descriptor took 2048
// tokens of 32 heads from 73.8 to 60.2 us (2 x 333 tokens, 64 heads over 8, 22.2 to 20.2). A block's K tile arrives by DMA (16-byte chunk p of row r holds the row's chunk
// p ^ (r % 16)), its V tile through registers, transposed four keys at a time; both go into the buffer
// that the tile after the current one reads.
#include <algorithm>

#include "nq_common.h"

namespace nq {
namespace {

constexpr int D = 128;
constexpr int kRowsPerBlock = 128;
constexpr int kKeys = 64;
constexpr float kSlack = 8.0f;
constexpr int kWholeTiles = 6;  // up to so many key tiles are not shared: the sums' way costs as much

struct AttnArgs {
    const uint16_t* q;
    const uint16_t* k;
    const uint16_t* v;
    int64_t q_stride, k_stride, v_stride;  // elements between tokens
    uint16_t* k_cache;
    uint16_t* v_cache;  // [batch][kv_heads][max_len][128]
    const uint16_t* cos;
    const uint16_t* sin;  // [tokens][128]
    const int64_t* positions;
    uint16_t* out;  // [batch][tokens][heads * 128]
    int batch, tokens, kv_heads, groups, max_len;
    float scale;  // times log2(e)
    float* part_o;  // [splits][batch * kv_heads * tokens * groups][128], where the keys are split
    float* part_ml;  // the same rows' {maximum, sum}
    int splits;
};

// Eight elements of a head and their rotary partners (d and d + 64): T(T(x cos) + T(rotate_half(x) sin)).
template <typename T>
__device__ inline void rotate8(u32x4& lo, u32x4& hi, const u32x4& c0, const u32x4& s0, const u32x4& c1, const u32x4& s1) {
#pragma clang fp contract(off)
    uint32_t a[4] = {lo.x, lo.y, lo.z, lo.w}, b[4] = {hi.x, hi.y, hi.z, hi.w};
    const uint32_t ca[4] = {c0.x, c0.y, c0.z, c0.w}, sa[4] = {s0.x, s0.y, s0.z, s0.w};
    const uint32_t cb[4] = {c1.x, c1.y, c1.z, c1.w}, sb[4] = {s1.x, s1.y, s1.z, s1.w};
#pragma unroll
    for (int w = 0; w < 4; ++w) {
        uint32_t ra = 0, rb = 0;
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            auto part = [&](uint32_t v) { return T::to_float(static_cast<uint16_t>(v >> (16 * h))); };
            auto round = [](float f) { return T::to_float(T::from_float(f)); };
            const float x0 = part(a[w]), x1 = part(b[w]), n1 = part(b[w] ^ 0x80008000u);  // n1 = -x1
            const uint16_t r0 = T::from_float(round(x0 * part(ca[w])) + round(n1 * part(sa[w])));
            const uint16_t r1 = T::from_float(round(x1 * part(cb[w])) + round(x0 * part(sb[w])));
            ra |= static_cast<uint32_t>(r0) << (16 * h);
            rb |= static_cast<uint32_t>(r1) << (16 * h);
        }
        a[w] = ra;
        b[w] = rb;
    }
    lo = u32x4{a[0], a[1], a[2], a[3]};
    hi = u32x4{b[0], b[1], b[2], b[3]};
}

__device__ inline const u32x4* vec(const uint16_t* p) { return reinterpret_cast<const u32x4*>(p); }

// Sixteen threads per (sequence, token, kv head): eight rotate 16 elements of the key each, eight copy 16 of
// the value.
template <typename T>
__global__ __launch_bounds__(256) void kv_rows_kernel(const AttnArgs a) {
    const int64_t id = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
    const int part = static_cast<int>(id & 15);
    const int64_t row = id >> 4;  // (b * tokens + t) * kv_heads + head
    if (row >= static_cast<int64_t>(a.batch) * a.tokens * a.kv_heads) return;
    const int64_t bt = row / a.kv_heads;
    const int head = static_cast<int>(row - bt * a.kv_heads);
    const int64_t b = bt / a.tokens;
    const int t = static_cast<int>(bt - b * a.tokens);
    const int64_t p = a.positions[t];
    if (p < 0 || p >= a.max_len) return;
    const size_t at = ((static_cast<size_t>(b) * a.kv_heads + head) * a.max_len + static_cast<size_t>(p)) * D;
    if (part < 8) {
        const uint16_t* src = a.k + bt * a.k_stride + head * D + 8 * part;
        const size_t tab = static_cast<size_t>(t) * D + 8 * part;
        u32x4 lo = *vec(src), hi = *vec(src + 64);
        rotate8<T>(lo, hi, *vec(a.cos + tab), *vec(a.sin + tab), *vec(a.cos + tab + 64), *vec(a.sin + tab + 64));
        uint16_t* dst = a.k_cache + at + 8 * part;
        *reinterpret_cast<u32x4*>(dst) = lo;
        *reinterpret_cast<u32x4*>(dst + 64) = hi;
    } else {
        const uint16_t* src = a.v + bt * a.v_stride + head * D + 16 * (part - 8);
        uint16_t* dst = a.v_cache + at + 16 * (part - 8);
        const u32x4 v0 = *vec(src), v1 = *vec(src + 8);
        *reinterpret_cast<u32x4*>(dst) = v0;
        *reinterpret_cast<u32x4*>(dst + 8) = v1;
    }
}

// Swizzle of the V^T tile (128 rows of 64 keys): the 16-byte chunk of row d that holds keys chunk ch. Reads
// take 16 consecutive rows at one ch; a transposing write takes rows 8 apart at one parity.
__device__ inline int vswz(int d) { return ((d >> 1) ^ (d >> 4)) & 7; }

template <typename T>
__device__ inline uint32_t pack2(float a, float b) {
    return static_cast<uint32_t>(T::from_float(a)) | (static_cast<uint32_t>(T::from_float(b)) << 16);
}

// kPart: a block takes one of a.splits shares of its rows' key tiles and leaves sums for attn_join_kernel.
template <typename T, int KS, bool kPart>
__global__ __launch_bounds__(256 * KS) __attribute__((amdgpu_waves_per_eu(2))) void prefill_attn_kernel(const AttnArgs a) {
    static_assert(KS == 1 || (KS == 2 && !kPart), "one or two groups of waves");
    __shared__ __attribute__((aligned(16))) uint16_t ksall[KS][2][kKeys * D];
    __shared__ __attribute__((aligned(16))) uint16_t vtall[KS][2][D * kKeys];
    __shared__ int lims[4];
    const int grp = KS == 1 ? 0 : __builtin_amdgcn_readfirstlane(threadIdx.x >> 8);  // key group
    const int t = static_cast<int>(threadIdx.x) & 255;
    auto& ks = ksall[grp];
    auto& vt = vtall[grp];
    const int lane = t & 63;
    const int wave = __builtin_amdgcn_readfirstlane(t >> 6);  // of its group
    const int c = lane & 31;
    const int kg = lane >> 5;
    const int heads = a.batch * a.kv_heads;
    // Row tiles in order of falling length, the longest blocks first. A grid that is resident at once (two
    // blocks a CU) has no later blocks to fill in behind the short ones: its second half goes the other
    // way round, so that a CU gets a long block and a short one.
    const int n_tiles = static_cast<int>(gridDim.x) / heads;  // (blockIdx.y: the share of the keys)
    const int order = static_cast<int>(blockIdx.x) / heads;
    const int tile = KS == 1 && gridDim.x <= 512u && 2 * order >= n_tiles ? order - (n_tiles + 1) / 2 : n_tiles - 1 - order;
    const int bh = static_cast<int>(blockIdx.x) % heads;
    const int b = bh / a.kv_heads;
    const int kvh = bh - b * a.kv_heads;
    const int rows = a.tokens * a.groups;
    const int R0 = tile * kRowsPerBlock + 32 * wave;
    const size_t q_row0 = static_cast<size_t>(b) * a.tokens;

    // the wave's queries, rotated: lane (c, kg) holds row R0 + c, dimensions 16 kt + 8 kg .. +7
    const int R = min(R0 + c, rows - 1);
    const int tok = R / a.groups;
    const int64_t p64 = a.positions[tok];
    const int lim = R0 + c < rows ? static_cast<int>(min<int64_t>(max<int64_t>(p64, -1), a.max_len - 1)) : -1;
    u32x4 qf[8];
    {
        const uint16_t* src = a.q + (q_row0 + tok) * a.q_stride + (kvh * a.groups + R - tok * a.groups) * D + 8 * kg;
#pragma unroll
        for (int kt = 0; kt < 8; ++kt) qf[kt] = *vec(src + 16 * kt);
        const size_t tab = static_cast<size_t>(tok) * D + 8 * kg;
#pragma unroll
        for (int kt = 0; kt < 4; ++kt)
            rotate8<T>(qf[kt], qf[kt + 4], *vec(a.cos + tab + 16 * kt), *vec(a.sin + tab + 16 * kt),
                       *vec(a.cos + tab + 16 * kt + 64), *vec(a.sin + tab + 16 * kt + 64));
    }
    // a positive factor, so that the largest product is the largest score: the queries take a negative
    // factor's sign, and are zero for a factor of zero
    const float scale = a.scale == 0.0f ? 1.0f : fabsf(a.scale);
    if (!(a.scale > 0.0f)) {
        const uint32_t keep = a.scale == 0.0f ? 0u : 0xffffffffu, flip = a.scale < 0.0f ? 0x80008000u : 0u;
#pragma unroll
        for (int kt = 0; kt < 8; ++kt)
            qf[kt] = u32x4{(qf[kt].x ^ flip) & keep, (qf[kt].y ^ flip) & keep, (qf[kt].z ^ flip) & keep,
                           (qf[kt].w ^ flip) & keep};
    }
    // the last visible position of the wave's rows and of the block's, and the first row's
    int wmax = lim, wmin = R0 + c < rows ? lim : a.max_len;
#pragma unroll
    for (int off = 16; off > 0; off >>= 1) {
        wmax = max(wmax, __shfl_xor(wmax, off, 64));
        wmin = min(wmin, __shfl_xor(wmin, off, 64));
    }
    wmax = __builtin_amdgcn_readfirstlane(wmax);
    wmin = __builtin_amdgcn_readfirstlane(wmin);
    if (grp == 0 && lane == 0) lims[wave] = wmax;
    __syncthreads();
    const int last = __builtin_amdgcn_readfirstlane(max(max(lims[0], lims[1]), max(lims[2], lims[3])));
    int tiles = last / kKeys + 1;  // one (all masked) where every position is below 0
    int it0 = 0;
    bool whole = !kPart;  // this block takes all of its rows' keys
    if (kPart) {
        whole = tiles <= kWholeTiles;
        if (whole && blockIdx.y > 0) return;
        const int share = whole ? tiles : (tiles + a.splits - 1) / a.splits;
        it0 = min(static_cast<int>(blockIdx.y) * share, tiles);
        tiles = min(share, tiles - it0);  // none in some last shares
    }

    const size_t head = static_cast<size_t>(bh) * a.max_len * D;
    const uint16_t* kbase = a.k_cache + head;
    // values past the block's last visible position load zeros
    const rsrc_t v_rs = make_rsrc(a.v_cache + head, static_cast<uint32_t>(last + 1) * (D * 2u));
    const uint32_t lk = __builtin_amdgcn_readfirstlane(lds_addr(&ks[0][0]) + static_cast<uint32_t>(wave) * 1024u);
    auto issue_k = [&](int it, int buf) {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int r = j * 16 + (t >> 4);
            const uint32_t row = static_cast<uint32_t>(min(it * kKeys + r, a.max_len - 1));
            dma16_lds(kbase, row * (D * 2u) + 16u * static_cast<uint32_t>((t & 15) ^ (r & 15)),
                      lk + static_cast<uint32_t>(buf) * (kKeys * D * 2u) + static_cast<uint32_t>(j) * 4096u);
        }
    };
    // thread (kq, dq) transposes keys 4 kq .. +3 by dimensions 8 dq .. +7
    const int kq = t >> 4, dq = t & 15;
    u32x4 vr[4];
    auto load_v = [&](int it) {
#pragma unroll
        for (int j = 0; j < 4; ++j)
            vr[j] = load_b128(v_rs, static_cast<uint32_t>(it * kKeys + 4 * kq + j) * (D * 2u) + 16u * static_cast<uint32_t>(dq));
    };
    // the keys of a 16-key tile in P^T's order: quads 0 and 2 are lane group 0's, 1 and 3 lane group 1's
    const int vchunk = 2 * (kq >> 2) + (kq & 1), vhalf = (kq >> 1) & 1;
    auto store_v = [&](int buf) {
        const uint32_t r0[4] = {vr[0].x, vr[0].y, vr[0].z, vr[0].w}, r1[4] = {vr[1].x, vr[1].y, vr[1].z, vr[1].w};
        const uint32_t r2[4] = {vr[2].x, vr[2].y, vr[2].z, vr[2].w}, r3[4] = {vr[3].x, vr[3].y, vr[3].z, vr[3].w};
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const int w = e >> 1;
            // the low (or high) halves of two keys side by side
            const uint32_t sel = (e & 1) ? 0x07060302u : 0x05040100u;
            const uint2 v = uint2{__builtin_amdgcn_perm(r1[w], r0[w], sel), __builtin_amdgcn_perm(r3[w], r2[w], sel)};
            const int d = 8 * dq + e;
            *reinterpret_cast<uint2*>(&vt[buf][d * kKeys + 8 * (vchunk ^ vswz(d)) + 4 * vhalf]) = v;
        }
    };

    f32x16 o[4];
#pragma unroll
    for (int dt = 0; dt < 4; ++dt)
#pragma unroll
        for (int i = 0; i < 16; ++i) o[dt][i] = 0.0f;
    float m = -__builtin_huge_valf(), l = 0.0f;

    // group g takes tiles g, g + KS, ...; all groups run the rounds of the longest (the barriers are the
    // block's), a tile past the last one being loaded (keys clamped, values zero) and not computed
    const int rounds = (tiles + KS - 1) / KS;
    if (!kPart || rounds > 0) {
        load_v(it0 + grp);
        issue_k(it0 + grp, 0);
        wait_vmcnt<0>();
        store_v(0);
    }
    barrier_keep_dma();
    for (int round = 0; round < rounds; ++round) {
        const int it = it0 + round * KS + grp;
        const int buf = round & 1;
        const bool more = round + 1 < rounds;
        if (more) {
            load_v(it + KS);
            issue_k(it + KS, buf ^ 1);
        }
        __builtin_amdgcn_sched_barrier(0);
        const int key0 = it * kKeys;
        if (key0 <= wmax) {  // uniform over the wave
            f32x16 s[2];
#pragma unroll
            for (int h = 0; h < 2; ++h)
#pragma unroll
                for (int i = 0; i < 16; ++i) s[h][i] = 0.0f;
            const uint16_t* kb = &ks[buf][c * D];
            // operands are read four ahead of the four MFMAs that run; left to itself the compiler reads two and
            // waits for them
            u32x4 kf[2][4], vf[2][4];
            auto read_k = [&](int g) {
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    kf[g & 1][e] = *vec(kb + 32 * (e & 1) * D + 8 * ((2 * (2 * g + (e >> 1)) + kg) ^ (c & 15)));
            };
            auto read_v = [&](int kt) {
#pragma unroll
                for (int dt = 0; dt < 4; ++dt) {
                    const int d = 32 * dt + c;
                    vf[kt & 1][dt] = *vec(&vt[buf][d * kKeys + 8 * ((2 * kt + kg) ^ vswz(d))]);
                }
            };
            read_k(0);
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                if (g < 3) read_k(g + 1);
                else read_v(0);
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int e = 0; e < 4; ++e) s[e & 1] = mfma32x32x16<T>(kf[g & 1][e], qf[2 * g + (e >> 1)], s[e & 1]);
                __builtin_amdgcn_sched_barrier(0);
            }
            const bool masked = key0 + kKeys - 1 > wmin;
            if (masked) {
#pragma unroll
                for (int h = 0; h < 2; ++h)
#pragma unroll
                    for (int i = 0; i < 16; ++i)
                        if (key0 + 32 * h + 8 * (i >> 2) + 4 * kg + (i & 3) > lim) s[h][i] = -__builtin_huge_valf();
            }
            float mt = -__builtin_huge_valf();
#pragma unroll
            for (int h = 0; h < 2; ++h)
#pragma unroll
                for (int i = 0; i < 16; ++i) mt = fmaxf(mt, s[h][i]);
            mt = fmaxf(mt, __shfl_xor(mt, 32, 64)) * scale;
            // the reference point of the exponentials follows the running maximum only once that is 8 above
            // it: exponentials up to 2^8 round the same, and most tiles rescale nothing
            if (__any(mt > m + kSlack)) {
                const float mn = fmaxf(m, mt);
                const float alpha = __builtin_amdgcn_exp2f(m - (mn == -__builtin_huge_valf() ? 0.0f : mn));
                m = mn;
                l *= alpha;
#pragma unroll
                for (int dt = 0; dt < 4; ++dt)
#pragma unroll
                    for (int i = 0; i < 16; ++i) o[dt][i] *= alpha;
            }
            const float mu = m == -__builtin_huge_valf() ? 0.0f : m;  // a row with nothing visible yet
            float sum = 0.0f;
#pragma unroll
            for (int h = 0; h < 2; ++h)
#pragma unroll
                for (int i = 0; i < 16; ++i) {
                    s[h][i] = __builtin_amdgcn_exp2f(fmaf(s[h][i], scale, -mu));
                    sum += s[h][i];
                }
            l += sum;
            auto pack_p = [&](int kt) {
                const f32x16& p = s[kt >> 1];
                const int i0 = 8 * (kt & 1);
                return u32x4{pack2<T>(p[i0], p[i0 + 1]), pack2<T>(p[i0 + 2], p[i0 + 3]),
                             pack2<T>(p[i0 + 4], p[i0 + 5]), pack2<T>(p[i0 + 6], p[i0 + 7])};
            };
            u32x4 pf = pack_p(0);
#pragma unroll
            for (int kt = 0; kt < 4; ++kt) {
                if (kt < 3) read_v(kt + 1);
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int dt = 0; dt < 4; ++dt) o[dt] = mfma32x32x16<T>(vf[kt & 1][dt], pf, o[dt]);
                if (kt < 3) pf = pack_p(kt + 1);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        if (more) {
            wait_vmcnt<0>();
            store_v(buf ^ 1);
        }
        barrier_keep_dma();
    }
    if constexpr (KS == 2) {  // group 1's sums join group 0's through the K buffers, its m and l behind 32 KB of V's
        float* red = reinterpret_cast<float*>(&ksall[0][0][0]);
        float* stat = reinterpret_cast<float*>(&vtall[1][0][0]);
        static_assert(sizeof(ksall) >= 64 * 256 * 4, "the K buffers hold a group's sums");
        if (grp == 1) {
#pragma unroll
            for (int dt = 0; dt < 4; ++dt)
#pragma unroll
                for (int i = 0; i < 16; ++i) red[(16 * dt + i) * 256 + t] = o[dt][i];
            stat[t] = m;
            stat[256 + t] = l;
        }
        __syncthreads();
        if (grp == 1) return;
        const float m1 = stat[t];
        const float mn = fmaxf(m, m1);
        const float mu = mn == -__builtin_huge_valf() ? 0.0f : mn;
        const float a0 = __builtin_amdgcn_exp2f(m - mu), a1 = __builtin_amdgcn_exp2f(m1 - mu);
        l = l * a0 + stat[256 + t] * a1;
#pragma unroll
        for (int dt = 0; dt < 4; ++dt)
#pragma unroll
            for (int i = 0; i < 16; ++i) o[dt][i] = o[dt][i] * a0 + red[(16 * dt + i) * 256 + t] * a1;
    }
    l += __shfl_xor(l, 32, 64);
    if constexpr (kPart) {  // the sums as they are, 16 bytes a lane
        if (R0 + c < rows) {
            const size_t row = (static_cast<size_t>(blockIdx.y) * heads + bh) * static_cast<size_t>(rows) + (R0 + c);
            // a sum of -1: the row is done
            if (kg == 0) *reinterpret_cast<float2*>(a.part_ml + 2 * row) = whole ? float2{0.0f, -1.0f} : float2{m, l};
            if (tiles > 0 && !whole) {
#pragma unroll
                for (int dt = 0; dt < 4; ++dt)
#pragma unroll
                    for (int g4 = 0; g4 < 4; ++g4)
                        *reinterpret_cast<f32x4*>(a.part_o + row * D + 32 * dt + 8 * g4 + 4 * kg) =
                            f32x4{o[dt][4 * g4], o[dt][4 * g4 + 1], o[dt][4 * g4 + 2], o[dt][4 * g4 + 3]};
            }
        }
        if (!whole) return;
    }
    const float inv = 1.0f / l;

    // the wave's rows through LDS (its 8 KB of the V buffers, 16-byte chunk ch of row r at ch ^ (r % 16)),
    // then whole 256-byte rows to memory
    uint16_t* ob = &vtall[0][0][0] + wave * 4096;
#pragma unroll
    for (int dt = 0; dt < 4; ++dt)
#pragma unroll
        for (int g4 = 0; g4 < 4; ++g4)
            *reinterpret_cast<uint2*>(ob + c * D + 8 * ((4 * dt + g4) ^ (c & 15)) + 4 * kg) =
                uint2{pack2<T>(o[dt][4 * g4] * inv, o[dt][4 * g4 + 1] * inv),
                      pack2<T>(o[dt][4 * g4 + 2] * inv, o[dt][4 * g4 + 3] * inv)};
#pragma unroll
    for (int j = 0; j < 8; ++j) {
        const int r = 4 * j + (lane >> 4);
        const int ch = lane & 15;
        const u32x4 v = *vec(ob + r * D + 8 * (ch ^ (r & 15)));
        if (R0 + r < rows) {
            const int tk = (R0 + r) / a.groups;
            const size_t at = ((q_row0 + tk) * (a.kv_heads * a.groups) + kvh * a.groups + (R0 + r - tk * a.groups)) * D;
            *reinterpret_cast<u32x4*>(a.out + at + 8 * ch) = v;
        }
    }
}

// out = T(sum_s o_s 2^(m_s - M) / sum_s l_s 2^(m_s - M)), M the largest m_s: 32 threads a row, four dimensions each.
// Bound by latency: eight shares' sums are loaded together. A share without keys has m = -inf and l = 0, and no o.
template <typename T>
__global__ __launch_bounds__(256) void attn_join_kernel(const AttnArgs a) {
    const int rows = a.tokens * a.groups;
    const int64_t total = static_cast<int64_t>(a.batch) * a.kv_heads * rows;
    const int64_t row = static_cast<int64_t>(blockIdx.x) * 8 + (threadIdx.x >> 5);
    const int d = 4 * static_cast<int>(threadIdx.x & 31);
    if (row >= total) return;
    if (a.part_ml[2 * row + 1] == -1.0f) return;  // (of share 0)
    float M = -__builtin_huge_valf(), L = 0.0f;
    f32x4 O = f32x4{0.f, 0.f, 0.f, 0.f};
    constexpr int kAhead = 8;
    for (int s0 = 0; s0 < a.splits; s0 += kAhead) {
        float2 ml[kAhead];
        f32x4 o[kAhead];
#pragma unroll
        for (int i = 0; i < kAhead; ++i) {
            const int64_t at = min(s0 + i, a.splits - 1) * total + row;
            ml[i] = *reinterpret_cast<const float2*>(a.part_ml + 2 * at);
            o[i] = *reinterpret_cast<const f32x4*>(a.part_o + at * D + d);
        }
        float bm = M;
#pragma unroll
        for (int i = 0; i < kAhead; ++i) bm = fmaxf(bm, ml[i].x);  // a share taken twice changes nothing here
        const float mu = bm == -__builtin_huge_valf() ? 0.0f : bm;
        const float keep = __builtin_amdgcn_exp2f(M - mu);
        L *= keep;
        O = f32x4{O.x * keep, O.y * keep, O.z * keep, O.w * keep};
#pragma unroll
        for (int i = 0; i < kAhead; ++i) {
            const bool none = s0 + i >= a.splits || (ml[i].x == -__builtin_huge_valf() && ml[i].y == 0.0f);
            const float f = __builtin_amdgcn_exp2f(ml[i].x - mu);
            L = none ? L : fmaf(ml[i].y, f, L);
            O = none ? O : f32x4{fmaf(o[i].x, f, O.x), fmaf(o[i].y, f, O.y), fmaf(o[i].z, f, O.z), fmaf(o[i].w, f, O.w)};
        }
        M = bm;
    }
    const float inv = 1.0f / L;
    const int64_t bh = row / rows;
    const int R = static_cast<int>(row - bh * rows);
    const int64_t b = bh / a.kv_heads;
    const int kvh = static_cast<int>(bh - b * a.kv_heads);
    const int tok = R / a.groups;
    const size_t at = ((static_cast<size_t>(b) * a.tokens + tok) * (a.kv_heads * a.groups) + kvh * a.groups + (R - tok * a.groups)) * D;
    *reinterpret_cast<uint2*>(a.out + at + d) = uint2{pack2<T>(O.x * inv, O.y * inv), pack2<T>(O.z * inv, O.w * inv)};
}

// Two groups of waves share a block's keys where the grid leaves a CU one block at most and its longest block
// walks over twelve tiles or more (the host does not know the positions, only that the last token sees at
// least the others): both launches, fp16, us, one group / two: 32 heads at 1000 tokens 43.1 / 40.4, 16 at 2000
// 62.2 / 53.5, 8 at 2000 57.6 / 48.2. Shorter chains do not pay for the joining of the groups (32 heads at 64
// tokens 12.7 / 15.5, two sequences of 512 32.8 / 33.5), and with two blocks to a CU these overlap better than
// two groups that meet at one barrier (32 heads at 2048 tokens, this launch alone, 60.2 / 62.5; 336 blocks of
// grouped heads 20.2 / 27.3).
constexpr int64_t kSplitBlocks = 256, kSplitTokens = 768;

// A few tokens on a long context are a few blocks with a long walk each, 1.2 us a tile, where the torch ops, slower
// otherwise, have the whole chip: their keys are shared over the grid, up to two blocks a CU, from caches of 4096 positions
// on (the host does not know how much of one is filled) and at least 512 positions a share. All launches, us, torch
// ops, whole, shared: 4 tokens of 8 heads over 2 after 29625 178, 567, 36; 2 tokens of 32 heads after 19239 236, 380, 66.
// A short context pays the join's launch: 2 to 64 tokens alone in such a cache 13-14 whole, 15 shared, torch ops 100-500.
// More tokens were never slower than the torch ops, and keep one launch.
constexpr int64_t kPartTokens = 64, kPartBlocks = 512, kPartKeys = 4096, kPartShare = 512, kPartMax = 32;
int prefill_splits(int64_t batch, int64_t tokens, int64_t kv_heads, int64_t groups, int64_t max_len) {
    const int64_t blocks = ceil_div(tokens * groups, kRowsPerBlock) * batch * kv_heads;
    if (blocks <= 0 || tokens > kPartTokens || max_len < kPartKeys) return 1;
    return static_cast<int>(std::max<int64_t>(1, std::min({kPartBlocks / blocks, max_len / kPartShare, kPartMax})));
}

template <typename T>
void launch_prefill(const AttnArgs& a, hipStream_t st) {
    const int64_t kv_threads = static_cast<int64_t>(a.batch) * a.tokens * a.kv_heads * 16;
    kv_rows_kernel<T><<<dim3(static_cast<unsigned>(ceil_div(kv_threads, 256))), 256, 0, st>>>(a);
    const int64_t tiles = ceil_div(static_cast<int64_t>(a.tokens) * a.groups, kRowsPerBlock);
    const int64_t blocks = tiles * a.batch * a.kv_heads;
    if (a.splits > 1) {
        prefill_attn_kernel<T, 1, true>
            <<<dim3(static_cast<unsigned>(blocks), static_cast<unsigned>(a.splits)), 256, 0, st>>>(a);
        const int64_t rows = static_cast<int64_t>(a.batch) * a.kv_heads * a.tokens * a.groups;
        attn_join_kernel<T><<<dim3(static_cast<unsigned>(ceil_div(rows, 8))), 256, 0, st>>>(a);
    } else if (blocks <= kSplitBlocks && a.tokens >= kSplitTokens) {
        prefill_attn_kernel<T, 2, false><<<dim3(static_cast<unsigned>(blocks)), 512, 0, st>>>(a);
    } else {
        prefill_attn_kernel<T, 1, false><<<dim3(static_cast<unsigned>(blocks)), 256, 0, st>>>(a);
    }
}

}  // namespace
}  // namespace nq

using namespace nq;

extern "C" {

size_t nq_attention_prefill_workspace_bytes(int64_t batch, int64_t tokens, int64_t heads, int64_t kv_heads, int64_t head_dim,
                                            int64_t max_len) {
    if (batch <= 0 || tokens <= 0 || heads <= 0 || kv_heads <= 0 || head_dim != D || heads % kv_heads || tokens > kPartTokens ||
        batch > INT32_MAX || heads > INT32_MAX || max_len > (int64_t{1} << 22))
        return 0;
    const int splits = prefill_splits(batch, tokens, kv_heads, heads / kv_heads, max_len);
    return splits > 1 ? static_cast<size_t>(splits) * batch * tokens * heads * (D + 2) * sizeof(float) : 0;
}

int nq_attention_prefill(int dtype, const void* q, int64_t q_stride, const void* k, int64_t k_stride, const void* v,
                         int64_t v_stride, void* k_cache, void* v_cache, const void* rope_cos, const void* rope_sin,
                         const int64_t* positions, void* out, int64_t batch, int64_t tokens, int64_t heads,
                         int64_t kv_heads, int64_t head_dim, int64_t max_len, float scaling, nq_stream_t stream) {
    return nq_attention_prefill_ws(dtype, q, q_stride, k, k_stride, v, v_stride, k_cache, v_cache, rope_cos, rope_sin, positions,
                                   out, batch, tokens, heads, kv_heads, head_dim, max_len, scaling, nullptr, 0, stream);
}

int nq_attention_prefill_ws(int dtype, const void* q, int64_t q_stride, const void* k, int64_t k_stride, const void* v,
                            int64_t v_stride, void* k_cache, void* v_cache, const void* rope_cos, const void* rope_sin,
                            const int64_t* positions, void* out, int64_t batch, int64_t tokens, int64_t heads,
                            int64_t kv_heads, int64_t head_dim, int64_t max_len, float scaling, void* workspace,
                            size_t workspace_bytes, nq_stream_t stream) {
    const char* name = "nq_attention_prefill";
    if (dtype != NQ_F16 && dtype != NQ_BF16) return fail(NQ_ERR_DTYPE, "%s: unsupported dtype %d", name, dtype);
    if (batch < 0 || tokens < 0 || heads <= 0 || kv_heads <= 0 || max_len <= 0)
        return fail(NQ_ERR_INVALID_ARGUMENT, "%s: bad sizes", name);
    if (head_dim != D || heads % kv_heads)
        return fail(NQ_ERR_UNSUPPORTED, "%s: needs head_dim %d and whole query groups per kv head", name, D);
    if (q_stride < heads * D || k_stride < kv_heads * D || v_stride < kv_heads * D || q_stride % 8 || k_stride % 8 ||
        v_stride % 8)
        return fail(NQ_ERR_SHAPE, "%s: token strides must hold the heads and be multiples of 8", name);
    if (max_len > (int64_t{1} << 22) || tokens * heads > INT32_MAX / 2 || batch * kv_heads > INT32_MAX / 2 ||
        batch * tokens * kv_heads > (int64_t{1} << 30) ||
        ceil_div(tokens * (heads / kv_heads), kRowsPerBlock) * batch * kv_heads > INT32_MAX / 2)
        return fail(NQ_ERR_UNSUPPORTED, "%s: sizes too large", name);
    if (batch == 0 || tokens == 0) return NQ_OK;
    if (!q || !k || !v || !k_cache || !v_cache || !rope_cos || !rope_sin || !positions || !out)
        return fail(NQ_ERR_INVALID_ARGUMENT, "%s: null pointer", name);
    for (const void* p : {q, k, v, static_cast<const void*>(k_cache), static_cast<const void*>(v_cache), rope_cos,
                          rope_sin, static_cast<const void*>(out)})
        if (!aligned(p, 16)) return fail(NQ_ERR_ALIGNMENT, "%s: tensors must be 16-byte aligned", name);
    if (!aligned(positions, 8)) return fail(NQ_ERR_ALIGNMENT, "%s: positions must be 8-byte aligned", name);
    if (!aligned(workspace, 16)) return fail(NQ_ERR_ALIGNMENT, "%s: workspace must be 16-byte aligned", name);
    AttnArgs a{};
    a.q = static_cast<const uint16_t*>(q);
    a.k = static_cast<const uint16_t*>(k);
    a.v = static_cast<const uint16_t*>(v);
    a.q_stride = q_stride;
    a.k_stride = k_stride;
    a.v_stride = v_stride;
    a.k_cache = static_cast<uint16_t*>(k_cache);
    a.v_cache = static_cast<uint16_t*>(v_cache);
    a.cos = static_cast<const uint16_t*>(rope_cos);
    a.sin = static_cast<const uint16_t*>(rope_sin);
    a.positions = positions;
    a.out = static_cast<uint16_t*>(out);
    a.batch = static_cast<int>(batch);
    a.tokens = static_cast<int>(tokens);
    a.kv_heads = static_cast<int>(kv_heads);
    a.groups = static_cast<int>(heads / kv_heads);
    a.max_len = static_cast<int>(max_len);
    a.scale = scaling * 1.44269504088896340736f;  // exp(x) = exp2(x log2(e))
    const size_t need = nq_attention_prefill_workspace_bytes(batch, tokens, heads, kv_heads, head_dim, max_len);
    a.splits = 1;
    if (workspace && need > 0 && workspace_bytes >= need) {
        a.splits = prefill_splits(batch, tokens, kv_heads, a.groups, max_len);
        a.part_o = static_cast<float*>(workspace);
        a.part_ml = a.part_o + static_cast<size_t>(a.splits) * batch * tokens * heads * D;
    }
    if (dtype == NQ_F16) launch_prefill<F16>(a, as_stream(stream));
    else launch_prefill<BF16>(a, as_stream(stream));
    return check_launch(name);
}

}  // extern "C"
