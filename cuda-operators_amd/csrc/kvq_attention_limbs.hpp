// kvq_attention_limbs.hpp -- dense fp32 attention on gfx950's bf16 matrix cores:
// out = softmax(Q K^T / sqrt(d)) V for Q[M,d], K/V[N,d] (one head), the math
// of the reference's attention_online_launch (attention/softmax_new.cu:87-281),
// for any d up to 256.
//
// Every fp32 value x is three bf16 limbs, h = bf16(x), m = bf16(x - h),
// l = x - h - m: 8 + 8 + 8 significand bits with signs hold all 24 of a value
// from 2^-110 up, and the differences are exact.  A product keeps the six limb pairs down to 2^-16 of
// it (hh, hm, mh, mm, hl, lh); the dropped ones are below 2^-24, and bf16
// products are exact in the fp32 accumulators.  Six v_mfma_f32_16x16x32_bf16
// take 96 cycles where the eight v_mfma_f32_16x16x4_f32 of the same contraction
// take 256.
//
// A workgroup of W waves owns 16 QB W queries and one split of the keys, which
// it streams through LDS in 32-key tiles:
// * K and V rows are loaded as fp32 (one tile ahead, in registers), split into
//   limbs once per workgroup and stored as bf16 planes: K rows as they are, V
//   transposed (a row per dim, keys in the order of the P operand), so both
//   MFMA A operands are single 16-byte LDS reads.  Head dims below D arrive as
//   zeros from out-of-bounds buffer loads.  Row strides (2D + 16 and 80 bytes)
//   put the 16 rows of a read in distinct bank groups.
// * S^T = K Q^T per 16-key block: B = this wave's q limbs (registers, scaled by
//   softmax_scale * log2 e before the split).  hh accumulates apart from the
//   five smaller products.  C leaves lane l with keys 4g + i (g = l / 16) of
//   query l % 16.
// * online softmax per query, as exp2 of log2-unit scores; the probabilities of
//   keys 4g + i and 16 + 4g + i are the lane's 8 contraction slots of PV, so P
//   needs no data movement, only its limb split.
// * O^T += V^T P^T, six MFMAs per 16-dim block.
// An input that is not finite, or a product that overflows, leaves NaN or
// infinity in the wave's state (a limb of it is NaN), and values below 2^-110
// have fewer bits than 24 (bf16's subnormals end at 2^-133); a wave that sees the
// first, or rows where the second counts (kLimbMin), recomputes its queries in
// fp32 (attention_block16).
//
// Splits write the (m, l, acc) records that attention_merge combines.  Measured
// against the kernel on v_mfma_f32_16x16x4_f32 that this one replaced: M = N =
// 4096 d = 128 83.6 -> 49.6 us, d = 64 48.5 -> 34.4 us, M = 8192 N = 1000 d = 256
// 93.8 -> 60.2 us, M = N = 1024 d = 128 16.6 -> 14.8 us; and against
// attention_generic, M = 1000 N = 3001 d = 96: 2007 -> 20.1 us.  Error against 64
// bits at the first: 5.9e-7 -> 4.0e-7.  Of the 50 us, MFMAs are 20, K and V
// reads from LDS about 8, and the merge launch 4.9.
#pragma once

#include <math.h>

#include "kvq_attention.hpp"

namespace kvq {
namespace {

typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

constexpr int kLimbKeys = kAttnLimbTile;  // keys per LDS tile
constexpr float kLazyMax = 8.0f;          // log2 units a score may pass the softmax reference by
constexpr float kLimbMin = 0x1p-60f;      // rows of q, and outputs, all below it take fp32 products
constexpr int kLimbOob = INT_MIN;         // byte offset of a load that reads zeros (past every resource)

// The limbs of a pair of floats, packed: h, m and l of x in the low halves, of y in the high.
__device__ __forceinline__ void split_pair(float x, float y, unsigned& h, unsigned& m, unsigned& l) {
    h = __builtin_bit_cast(unsigned, bf16x2{static_cast<__bf16>(x), static_cast<__bf16>(y)});
    x -= __uint_as_float(h << 16);
    y -= __uint_as_float(h & 0xffff0000u);
    m = __builtin_bit_cast(unsigned, bf16x2{static_cast<__bf16>(x), static_cast<__bf16>(y)});
    x -= __uint_as_float(m << 16);
    y -= __uint_as_float(m & 0xffff0000u);
    // What is left has at most 8 significant bits: its high half is all of it.
    l = __builtin_amdgcn_perm(__float_as_uint(y), __float_as_uint(x), 0x07060302u);
}

__device__ __forceinline__ f32x4 mma(const uint4& a, const uint4& b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0,
                                                   0, 0);
}

// 16 queries from q0 over keys [k0, k1) by one wave on v_mfma_f32_16x16x4_f32:
// fp32 products in place of the limbs', the same state (o, m and the whole l,
// relative to the exact running max).  K, V and q come straight from
// memory, 16 keys at a time; elements past d and rows past k1 or M are zeros.
// It runs for the waves whose limbs do not hold their values, so it keeps few
// registers and no loads in flight over a block: 2-3 times the limb kernel's
// time if every wave takes it (M = N = 4096 d = 128 142 us, and 5920 with one
// query at a time in FMAs; M = 1000 N = 3001 d = 96 41 us, 1265).
template <int D>
__device__ __forceinline__ void attention_block16(const AttnArgs& a, int q0, int k0, int k1, f32x4 (&o)[D / 16], float& m,
                                                  float& l) {
    constexpr int NB = D / 16;
    const int lane = threadIdx.x & (kWave - 1);
    const int r = lane & 15;
    const int g = lane >> 4;
    const int d = a.d;
    // Row r of 16 rows, dims 16 j + 4 g + [0, 4): one contraction index of four steps.
    auto piece = [&](buf_rsrc rs, int j) {
        const int c = 16 * j + 4 * g;
        float4 x = __builtin_bit_cast(float4, buffer_load16(rs, c < d ? (r * d + c) * 4 : kLimbOob, 0));
        if (c + 1 >= d) x.y = 0.0f;
        if (c + 2 >= d) x.z = 0.0f;
        if (c + 3 >= d) x.w = 0.0f;
        return x;
    };
    const buf_rsrc qr = make_rsrc(a.q + static_cast<size_t>(q0) * d, static_cast<unsigned>(min(16, a.M - q0)) * d * 4u);
#pragma unroll
    for (int c = 0; c < NB; c++) o[c] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    m = -INFINITY;
    l = 0.0f;
#pragma unroll 1
    for (int t = k0; t < k1; t += 16) {
        const unsigned bytes = static_cast<unsigned>(min(16, k1 - t)) * d * 4u;
        const buf_rsrc kr = make_rsrc(a.k + static_cast<size_t>(t) * d, bytes);
        const buf_rsrc vr = make_rsrc(a.v + static_cast<size_t>(t) * d, bytes);
        f32x4 s = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int j = 0; j < NB; j++) {
            const float4 x = piece(kr, j);
            const float4 y = piece(qr, j);
            s = __builtin_amdgcn_mfma_f32_16x16x4f32(x.x, y.x * a.scale_log2, s, 0, 0, 0);
            s = __builtin_amdgcn_mfma_f32_16x16x4f32(x.y, y.y * a.scale_log2, s, 0, 0, 0);
            s = __builtin_amdgcn_mfma_f32_16x16x4f32(x.z, y.z * a.scale_log2, s, 0, 0, 0);
            s = __builtin_amdgcn_mfma_f32_16x16x4f32(x.w, y.w * a.scale_log2, s, 0, 0, 0);
        }
        // s[i]: score of key t + 4 g + i for query q0 + r.
#pragma unroll
        for (int i = 0; i < 4; i++) s[i] = t + 4 * g + i < k1 ? s[i] : -INFINITY;
        float mt = fmaxf(fmaxf(s[0], s[1]), fmaxf(s[2], s[3]));
        mt = fmaxf(mt, __shfl_xor(mt, 16));
        mt = fmaxf(mt, __shfl_xor(mt, 32));
        const float mn = fmaxf(m, mt);
        const float ms = mn == -INFINITY ? 0.0f : mn;
        const float alpha = fast_exp2(m - ms);
        m = mn;
        l *= alpha;
#pragma unroll
        for (int i = 0; i < 4; i++) {
            s[i] = fast_exp2(s[i] - ms);
            l += s[i];
        }
#pragma unroll
        for (int c = 0; c < NB; c++) {
            o[c] *= alpha;
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const int off = 16 * c + r < d ? ((4 * g + i) * d + 16 * c + r) * 4 : kLimbOob;
                const float v = __int_as_float(buffer_load4(vr, off, 0));
                o[c] = __builtin_amdgcn_mfma_f32_16x16x4f32(v, s[i], o[c], 0, 0, 0);
            }
        }
    }
    l += __shfl_xor(l, 16);
    l += __shfl_xor(l, 32);
}

template <int D, int W, int QB, int BUFS>
__global__ __launch_bounds__(W* kWave) __attribute__((amdgpu_waves_per_eu(D <= 32 ? 4 : W / 4))) void attention_limbs(
    const AttnArgs a) {  // (two workgroups per CU at D = 32, one otherwise)
    static_assert(D % 32 == 0, "whole 32-dim contraction steps");
    constexpr bool kPhased = W == 8 && BUFS == 2;
    constexpr int AK = kLimbKeys;
    constexpr int NS = D / 32;                // QK contraction steps
    constexpr int NB = D / 16;                // output blocks
    constexpr int KS = D + 8, VS = AK + 8;    // LDS row strides in bf16
    constexpr int BANDS = D / 32;             // 32-dim bands of a tile, one wave load each
    constexpr int NU = (BANDS + W / 2 - 1) / (W / 2);
    __shared__ __align__(16) unsigned short s_kt[BUFS][3 * AK * KS];
    __shared__ __align__(16) unsigned short s_vt[BUFS][3 * D * VS];
    static_assert(sizeof(s_kt) + sizeof(s_vt) <= 160 * 1024, "LDS");

    const int lane = threadIdx.x & (kWave - 1);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const int r = lane & 15;
    const int g = lane >> 4;
    const int d = a.d;
    const int split = blockIdx.y;
    const int q0 = blockIdx.x * (16 * QB * W) + wave * (16 * QB);
    const int k0 = split * a.chunk;
    const int k1 = attention_split_end(a.N, split, a.chunk);
    const int tiles = (k1 - k0 + AK - 1) / AK;

    // The first half of the waves loads and stores K tiles, the second V tiles,
    // a 32-dim band at a time: lane (kq, c) takes rows 4kq .. 4kq+3, dims
    // 4c .. 4c+3 of the band (128-byte row segments; the transposing V stores of
    // 32 lanes cover all 64 banks once).  Rows past the split's end and dims past
    // d read zeros.
    const bool is_v = wave >= W / 2;
    const int hwave = is_v ? wave - W / 2 : wave;
    const float* const src = is_v ? a.v : a.k;
    const int kq = lane >> 3;
    float4 pre[NU][4];
    auto load_tile = [&](int t) {
        const int t0 = k0 + t * AK;
        const buf_rsrc rs =
            make_rsrc(src + static_cast<size_t>(t0) * d, static_cast<unsigned>(min(AK, k1 - t0)) * d * 4u);
#pragma unroll
        for (int j = 0; j < NU; j++) {
            const int band = hwave + j * (W / 2);
            if (BANDS % (W / 2) != 0 && band >= BANDS) break;
            const int c = 8 * band + (lane & 7);
            const int off = 4 * c < d ? (4 * kq * d + 4 * c) * 4 : kLimbOob;
#pragma unroll
            for (int i = 0; i < 4; i++)
                pre[j][i] = __builtin_bit_cast(float4, buffer_load16(rs, off + i * d * 4, 0));
            if ((d & 3) != 0) {  // the last piece runs into the next row
                const int n = d - 4 * c;
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    if (n < 2) pre[j][i].y = 0.0f;
                    if (n < 3) pre[j][i].z = 0.0f;
                    if (n < 4) pre[j][i].w = 0.0f;
                }
            }
        }
    };
    auto store_tile = [&](int t) {
        unsigned short* const s_k = s_kt[t % BUFS];
        unsigned short* const s_v = s_vt[t % BUFS];
#pragma unroll
        for (int j = 0; j < NU; j++) {
            const int band = hwave + j * (W / 2);
            if (BANDS % (W / 2) != 0 && band >= BANDS) break;
            const int c = 8 * band + (lane & 7);
            if (!is_v) {
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    uint2 h, m, l;
                    split_pair(pre[j][i].x, pre[j][i].y, h.x, m.x, l.x);
                    split_pair(pre[j][i].z, pre[j][i].w, h.y, m.y, l.y);
                    unsigned short* const p = s_k + (4 * kq + i) * KS + 4 * c;
                    *reinterpret_cast<uint2*>(p) = h;
                    *reinterpret_cast<uint2*>(p + AK * KS) = m;
                    *reinterpret_cast<uint2*>(p + 2 * AK * KS) = l;
                }
            } else {
                // Keys 4kq .. 4kq+3 of a dim: slots 4 (kq / 4) .. of the 8 that lane group kq % 4 contracts.
                const int slot = 8 * (kq & 3) + 4 * (kq >> 2);
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    float x[4];
#pragma unroll
                    for (int i = 0; i < 4; i++)
                        x[i] = e == 0 ? pre[j][i].x : e == 1 ? pre[j][i].y : e == 2 ? pre[j][i].z : pre[j][i].w;
                    uint2 h, m, l;
                    split_pair(x[0], x[1], h.x, m.x, l.x);
                    split_pair(x[2], x[3], h.y, m.y, l.y);
                    unsigned short* const p = s_v + (4 * c + e) * VS + slot;
                    *reinterpret_cast<uint2*>(p) = h;
                    *reinterpret_cast<uint2*>(p + D * VS) = m;
                    *reinterpret_cast<uint2*>(p + 2 * D * VS) = l;
                }
            }
        }
    };
    load_tile(0);

    // This wave's q^T operands: lane holds limbs of dims 32 s + 8 g + [0, 8) of query q0 + 16 b + r, scaled.
    uint4 qh[QB][NS], qm[QB][NS], ql[QB][NS];
    const int qb0 = blockIdx.x * (16 * QB * W);
    const buf_rsrc qrs = make_rsrc(a.q + static_cast<size_t>(qb0) * d,
                                   static_cast<unsigned>(min(16 * QB * W, a.M - qb0)) * d * 4u);
#pragma unroll
    for (int b = 0; b < QB; b++) {
        const int row = (wave * (16 * QB) + 16 * b + r) * d;  // rows past M read zeros
#pragma unroll
        for (int s = 0; s < NS; s++) {
            float x[8];
#pragma unroll
            for (int p = 0; p < 2; p++) {
                const int c = 32 * s + 8 * g + 4 * p;
                const float4 y = __builtin_bit_cast(float4, buffer_load16(qrs, c < d ? (row + c) * 4 : kLimbOob, 0));
                x[4 * p] = y.x * a.scale_log2;
                x[4 * p + 1] = c + 1 < d ? y.y * a.scale_log2 : 0.0f;
                x[4 * p + 2] = c + 2 < d ? y.z * a.scale_log2 : 0.0f;
                x[4 * p + 3] = c + 3 < d ? y.w * a.scale_log2 : 0.0f;
            }
            split_pair(x[0], x[1], qh[b][s].x, qm[b][s].x, ql[b][s].x);
            split_pair(x[2], x[3], qh[b][s].y, qm[b][s].y, ql[b][s].y);
            split_pair(x[4], x[5], qh[b][s].z, qm[b][s].z, ql[b][s].z);
            split_pair(x[6], x[7], qh[b][s].w, qm[b][s].w, ql[b][s].w);
        }
    }
    f32x4 o[QB][NB];
    float m[QB], l[QB];
#pragma unroll
    for (int b = 0; b < QB; b++) {
#pragma unroll
        for (int c = 0; c < NB; c++) o[b][c] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
        m[b] = -INFINITY;
        l[b] = 0.0f;
    }

    float sv[QB][8];  // sv[b][4 kb + i]: score of the tile's key 16 kb + 4 g + i, query 16 b + r
    uint4 ph[QB], pm[QB], pl[QB];
    struct Limbs {
        uint4 h, m, l;
    };
    // S^T of tile t.  Operands of the next step are read while one computes.
    auto scores = [&](int t) {
        const unsigned short* const s_k = s_kt[t % BUFS] + r * KS + 8 * g;
        auto read = [&](int n) {
            const unsigned short* const p = s_k + 16 * (n / NS) * KS + 32 * (n % NS);
            return Limbs{*reinterpret_cast<const uint4*>(p), *reinterpret_cast<const uint4*>(p + AK * KS),
                         *reinterpret_cast<const uint4*>(p + 2 * AK * KS)};
        };
        f32x4 hi[QB], lo[QB];
        Limbs x = read(0);
#pragma unroll
        for (int n = 0; n < 2 * NS; n++) {
            const Limbs nx = n + 1 < 2 * NS ? read(n + 1) : x;
            __builtin_amdgcn_sched_barrier(0);
            const int s = n % NS;
            if (s == 0) {
#pragma unroll
                for (int b = 0; b < QB; b++) hi[b] = lo[b] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
            }
#pragma unroll
            for (int b = 0; b < QB; b++) lo[b] = mma(x.l, qh[b][s], lo[b]);
#pragma unroll
            for (int b = 0; b < QB; b++) hi[b] = mma(x.h, qh[b][s], hi[b]);
#pragma unroll
            for (int b = 0; b < QB; b++) lo[b] = mma(x.h, ql[b][s], lo[b]);
#pragma unroll
            for (int b = 0; b < QB; b++) lo[b] = mma(x.m, qm[b][s], lo[b]);
#pragma unroll
            for (int b = 0; b < QB; b++) lo[b] = mma(x.m, qh[b][s], lo[b]);
#pragma unroll
            for (int b = 0; b < QB; b++) lo[b] = mma(x.h, qm[b][s], lo[b]);
            __builtin_amdgcn_sched_barrier(0);
            if (s == NS - 1) {
#pragma unroll
                for (int b = 0; b < QB; b++)
#pragma unroll
                    for (int i = 0; i < 4; i++) sv[b][4 * (n / NS) + i] = hi[b][i] + lo[b][i];
            }
            x = nx;
        }
    };
    auto softmax = [&](int t) {
        const int t0 = k0 + t * AK;
        if (t0 + AK > k1) {
#pragma unroll
            for (int j = 0; j < 8; j++) {
                const bool in = t0 + 16 * (j >> 2) + 4 * g + (j & 3) < k1;
#pragma unroll
                for (int b = 0; b < QB; b++) sv[b][j] = in ? sv[b][j] : -INFINITY;
            }
        }
        // m is a reference within 2^kLazyMax of the running max: it moves (and
        // the state is rescaled) only when some score of the wave passes it by
        // more, so most tiles need no cross-lane max.
        float mt[QB];
        bool grow = false;
#pragma unroll
        for (int b = 0; b < QB; b++) {
            mt[b] = sv[b][0];
#pragma unroll
            for (int j = 1; j < 8; j++) mt[b] = fmaxf(mt[b], sv[b][j]);
            grow |= mt[b] > m[b] + kLazyMax;
        }
        if (__builtin_amdgcn_ballot_w64(grow) != 0) {
#pragma unroll
            for (int b = 0; b < QB; b++) {
                float x = fmaxf(mt[b], __shfl_xor(mt[b], 16));
                x = fmaxf(x, __shfl_xor(x, 32));
                const float mn = fmaxf(m[b], x);
                const float alpha = mn == -INFINITY ? 1.0f : fast_exp2(m[b] - mn);
                m[b] = mn;
                l[b] *= alpha;
#pragma unroll
                for (int c = 0; c < NB; c++) o[b][c] *= alpha;
            }
        }
#pragma unroll
        for (int b = 0; b < QB; b++) {
            const float ms = m[b] == -INFINITY ? 0.0f : m[b];
#pragma unroll
            for (int j = 0; j < 8; j++) {
                sv[b][j] = fast_exp2(sv[b][j] - ms);
                l[b] += sv[b][j];
            }
            split_pair(sv[b][0], sv[b][1], ph[b].x, pm[b].x, pl[b].x);
            split_pair(sv[b][2], sv[b][3], ph[b].y, pm[b].y, pl[b].y);
            split_pair(sv[b][4], sv[b][5], ph[b].z, pm[b].z, pl[b].z);
            split_pair(sv[b][6], sv[b][7], ph[b].w, pm[b].w, pl[b].w);
        }
    };
    // O^T += V^T P^T of tile t.
    auto values = [&](int t) {
        const unsigned short* const s_v = s_vt[t % BUFS] + r * VS + 8 * g;
        auto read = [&](int c) {
            const unsigned short* const p = s_v + 16 * c * VS;
            return Limbs{*reinterpret_cast<const uint4*>(p), *reinterpret_cast<const uint4*>(p + D * VS),
                         *reinterpret_cast<const uint4*>(p + 2 * D * VS)};
        };
        Limbs x = read(0);
#pragma unroll
        for (int c = 0; c < NB; c++) {
            const Limbs nx = c + 1 < NB ? read(c + 1) : x;
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int b = 0; b < QB; b++) o[b][c] = mma(x.l, ph[b], o[b][c]);
#pragma unroll
            for (int b = 0; b < QB; b++) o[b][c] = mma(x.h, pl[b], o[b][c]);
#pragma unroll
            for (int b = 0; b < QB; b++) o[b][c] = mma(x.m, pm[b], o[b][c]);
#pragma unroll
            for (int b = 0; b < QB; b++) o[b][c] = mma(x.m, ph[b], o[b][c]);
#pragma unroll
            for (int b = 0; b < QB; b++) o[b][c] = mma(x.h, pm[b], o[b][c]);
#pragma unroll
            for (int b = 0; b < QB; b++) o[b][c] = mma(x.h, ph[b], o[b][c]);
            __builtin_amdgcn_sched_barrier(0);
            x = nx;
        }
    };

    store_tile(0);
    if (1 < tiles) load_tile(1);
    __syncthreads();
    if constexpr (kPhased) {
        // Two phases per tile, a barrier after each: matrix cores (PV of tile
        // t - 1, QK of tile t), then vector ALU (softmax of t, limbs of the next
        // tile).  The V waves run one phase behind the K waves, so each SIMD's
        // two waves (one of each half) use different units.  K wave phases: 2t
        // and 2t + 1; V waves: 2t + 1 and 2t + 2.
        // * K tile t + 1 is stored in phase 2t + 1: its buffer's last readers
        //   (QK of t - 1) were the V waves in phase 2t - 1, its first reader is a
        //   K wave in phase 2t + 2.
        // * V tile t + 1 is stored in phase 2t + 2: its buffer's last readers (PV
        //   of t - 1) were the V waves in phase 2t + 1, its first reader is a K
        //   wave in phase 2t + 4.
        // Every wave passes 2 * tiles + 1 barriers.
        if (is_v) __syncthreads();
        for (int t = 0; t < tiles; t++) {
            if (t > 0) values(t - 1);
            scores(t);
            __syncthreads();
            softmax(t);
            if (t + 1 < tiles) {
                store_tile(t + 1);
                if (t + 2 < tiles) load_tile(t + 2);
            }
            __syncthreads();
        }
        values(tiles - 1);
        if (!is_v) __syncthreads();
    } else {
        // One wave per SIMD, or (D > 128) one buffer.
        for (int t = 0; t < tiles; t++) {
            if (BUFS == 2 && t + 1 < tiles) {
                store_tile(t + 1);
                if (t + 2 < tiles) load_tile(t + 2);
            }
            scores(t);
            softmax(t);
            values(t);
            __syncthreads();
            if (BUFS == 1 && t + 1 < tiles) {
                store_tile(t + 1);
                if (t + 2 < tiles) load_tile(t + 2);
                __syncthreads();
            }
        }
    }

    // What the limbs cannot hold: NaN or infinity in the state, and values below
    // 2^-110, of which up to 2^-126 can be lost (a limb under bf16's subnormals).
    // That is nothing in an output row whose largest element is above kLimbMin
    // (weights sum to 1 or more), and nothing in the scores of a q row whose
    // largest is above kLimbMin and not above its reciprocal (or 0).  A row is
    // spread over four lane groups, whose ballots are folded.
    unsigned long long bad = 0;
    auto none = [](bool x) {  // rows for which no group has x, in the low 16 bits
        const unsigned long long y = __builtin_amdgcn_ballot_w64(x);
        return ~(y | y >> 16 | y >> 32 | y >> 48) & 0xffff;
    };
#pragma unroll
    for (int b = 0; b < QB; b++) {
        float top = 0.0f;
#pragma unroll
        for (int c = 0; c < NB; c++)
#pragma unroll
            for (int i = 0; i < 4; i++) top = max_or_nan(top, fabsf(o[b][c][i]));
        typedef unsigned short u16x2 __attribute__((ext_vector_type(2)));
        u16x2 qt = {0, 0};  // high limbs' magnitudes
#pragma unroll
        for (int s = 0; s < NS; s++)
#pragma unroll
            for (const unsigned x : {qh[b][s].x, qh[b][s].y, qh[b][s].z, qh[b][s].w})
                qt = __builtin_elementwise_max(qt, __builtin_bit_cast(u16x2, x & 0x7fff7fffu));
        const float qmax = __uint_as_float(static_cast<unsigned>(max(qt.x, qt.y)) << 16);
        bad |= __builtin_amdgcn_ballot_w64(!(top < INFINITY && l[b] < INFINITY && qmax <= 1.0f / kLimbMin)) |
               none(top >= kLimbMin) | (none(qmax >= kLimbMin) & ~none(qmax != 0.0f));
        l[b] += __shfl_xor(l[b], 16);
        l[b] += __shfl_xor(l[b], 32);
    }
    if (__builtin_expect(bad != 0, 0)) {
#pragma unroll
        for (int b = 0; b < QB; b++)
            if (q0 + 16 * b < a.M) attention_block16<D>(a, q0 + 16 * b, k0, k1, o[b], m[b], l[b]);
    }

    // The normalised output (one split) or the partial record of (split, query).
    const bool whole = a.splits == 1;
    const int ps = attention_record_dim(d);
#pragma unroll
    for (int b = 0; b < QB; b++) {
        const int q = q0 + 16 * b + r;
        if (q >= a.M) continue;
        const float inv = whole ? 1.0f / l[b] : 1.0f;
        float* const row = whole ? a.out + static_cast<size_t>(q) * d
                                 : a.part_acc + (static_cast<size_t>(split) * a.M + q) * ps;
        const int lim = whole ? d : ps;
#pragma unroll
        for (int c = 0; c < NB; c++) {
            const int dim = 16 * c + 4 * g;
            if ((lim & 3) == 0) {
                if (dim < lim)
                    *reinterpret_cast<float4*>(row + dim) =
                        make_float4(o[b][c][0] * inv, o[b][c][1] * inv, o[b][c][2] * inv, o[b][c][3] * inv);
            } else {
#pragma unroll
                for (int i = 0; i < 4; i++)
                    if (dim + i < lim) row[dim + i] = o[b][c][i] * inv;
            }
        }
        if (!whole && g == 0)
            *reinterpret_cast<float2*>(a.part_ml + (static_cast<size_t>(split) * a.M + q) * 2) = make_float2(m[b], l[b]);
    }
}

template <int D, int W, int QB>
void launch_limbs(const AttnArgs& a, hipStream_t stream) {
    constexpr int kBuf = 2 * 3 * (kLimbKeys * (D + 8) + D * (kLimbKeys + 8));
    constexpr int kBufs = 2 * kBuf <= 160 * 1024 ? 2 : 1;
    constexpr int kBlock = 16 * QB * W;
    const dim3 grid(static_cast<unsigned>((a.M + kBlock - 1) / kBlock), static_cast<unsigned>(a.splits));
    hipLaunchKernelGGL((attention_limbs<D, W, QB, kBufs>), grid, dim3(W * kWave), 0, stream, a);
}
template <int D>
void launch_limbs_d(const AttnArgs& a, hipStream_t stream) {
    if constexpr (D <= 128) {
        if (a.qblock == 256) {
            launch_limbs<D, 8, 2>(a, stream);
            return;
        }
    }
    if (a.qblock == 128) launch_limbs<D, 8, 1>(a, stream);
    else launch_limbs<D, 4, 1>(a, stream);
}
void launch_attention_limbs(const AttnArgs& a, hipStream_t stream) {  // without the merge
    if (a.d <= 32) launch_limbs_d<32>(a, stream);
    else if (a.d <= 64) launch_limbs_d<64>(a, stream);
    else if (a.d <= 96) launch_limbs_d<96>(a, stream);
    else if (a.d <= 128) launch_limbs_d<128>(a, stream);
    else if (a.d <= 192) launch_limbs_d<192>(a, stream);
    else launch_limbs_d<256>(a, stream);
}

}  // namespace
}  // namespace kvq
