// grouped_rows.hip - gfx950 expert products of many-token calls (gate/up + SwiGLU, down) on the int8 matrix cores
// for every pool format: Q8_0, Q4_K and KQ8 (Q2_K, Q3_K, Q5_K, Q6_K unpacked), src/qwen3.cpp:201-205.
//
// Work item = up to 16 MT pairs of one expert (permute_kernel's list, grouped.hip; 16-row products rather than 32 because
// a few hundred tokens leave each of 128 experts some 10 to 40 pairs, and products of rows past the last are wasted). A work-group stages the item's
// quantized activation rows in LDS once, whole rows, and meets at one barrier; after that each of its NW wavefronts
// streams the weight rows of its own two 16-row tiles (gate and up of 16 rows, or 32 down rows) from memory straight
// into registers, the next super-block requested before the current one is multiplied, and never waits for another
// wavefront again. The pool layout already is the operand layout: of a 32-value block, lane (kg, r) = (lane / 16,
// lane % 16) takes bytes 8 kg .. 8 kg + 7 of row r, and a wavefront's load covers 512 contiguous bytes.
//
// One v_mfma_i32_16x16x32_i8 (tokens x rows) is one 32-value block, the unit Q8_0 and Q4_K scale:
//   Q8_0  acc += d_x (d_w I). The product starts from the constant accumulator 0x4b400000, the bits of 1.5 2^23: its
//         int32 result read as a float is 1.5 2^23 + I exactly (|I| <= 516128), so one fma with the exact addend
//         -1.5 2^23 d_w gives d_w I rounded once, and a second one adds d_x of it: two VALU operations per output
//         and block instead of convert, multiply and fma. A super-block's eight blocks are summed on their own and
//         the super-blocks after that, as the GEMV kernels' threads do: one chain over the 64 blocks of K 2048 would
//         round 1.7 times as far from 64 bits (1.45e-7 of the result against 0.83e-7, and 0.80e-7 as it is).
//   Q4_K  isum += sc I (24-bit multiply-add, exact), imin on one v_mfma_f32_16x16x32_f16 per super-block over the split
//         group sums (exact integers, as in grouped.hip), then acc += d_x (d_w isum - dmin imin).
//   KQ8   scales per 16 values: two products per block, each seeing the tokens of one half of K and zeros for the
//         other (lanes of the other half read a zeroed LDS piece); isum as Q4_K. imin = sum m_g x as products of the
//         tokens with the mins spread over the block's bytes.
// Integer sums are those of ggml's vec_dot; only the f32 order over super-blocks differs.
//
// Bound: the expert bytes while an expert has a few pairs (64 tokens through a 30B-shaped Q2_K + Q3_K layer: 153 us for
// 717 MB of unpacked weights); past that the bytes of an expert's items, fetched about once (1.05 to 1.11 times the weights) at 3.5
// to 4.3 TB/s, beside VALU work that keeps the VALU half busy (512 Q8_0 tokens 51% and 45%, matrix cores 15% and 12%). Against the GEMV kernels, which served these calls
// before with dot products on the VALU and a work-group per expert however many pairs it had, on 30B-shaped layers on
// MI355X: 512 tokens Q8_0 630 -> 202 us a layer, 203 tokens Q4_K + Q6_K 329 -> 130, 64 tokens Q2_K + Q3_K 200 -> 153 (-> 134 with
// the weights' non-temporal loads of calls whose experts mostly have one item, GroupedParams::once).
#include "device.h"
#include "formats.h"
#include "kernels.h"

#include <algorithm>
#include <type_traits>

namespace lstk {
namespace {

typedef int i32x4 __attribute__((ext_vector_type(4)));
typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef __attribute__((address_space(3))) void lds_void;

constexpr int kRXcds = 8;
constexpr int kMagic = 0x4b400000;         // bits of 1.5 2^23
constexpr float kMagicF = 12582912.0f;

__device__ __forceinline__ i32x4 mfma8(uint2 a, uint2 b, i32x4 c) {
    return __builtin_amdgcn_mfma_i32_16x16x32_i8(__builtin_bit_cast(long, a), __builtin_bit_cast(long, b), c, 0, 0, 0);
}

// v as a value of this place: what is derived from it is formed here and not ahead of time, held in registers.
__device__ __forceinline__ unsigned here(unsigned v) {
    asm volatile("" : "+v"(v));
    return v;
}

// One 256-value super-block of a 16-row tile as the lane holds it: its share of the quants, and the rows' scales.
template <int WT>
struct TileQ {
    uint2 q[WT == kTypeQ4_K ? 4 : 8]; // 8 bytes per 32-value block (Q4_K: per pair of blocks)
};
template <int WT, bool MINS>
struct TileH {
    uint4 h;                                             // Q8_0: 8 fp16 scales; Q4_K: {d, dmin, 6-bit scales and mins}; KQ8: 16 int8 scales
    uint4 m[WT == kTypeKQ8 && MINS ? 1 : 0];             // KQ8: 16 mins
    float2 d[WT == kTypeKQ8 ? 1 : 0];                    // KQ8: d, dmin
};

// A weight load; NT: with the non-temporal hint (load_weights, device.h).
template <bool NT, typename T>
__device__ __forceinline__ T load_w(const uint8_t *p) {
    typedef unsigned uv __attribute__((ext_vector_type(sizeof(T) / 4)));
    const uv *q = reinterpret_cast<const uv *>(p);
    return __builtin_bit_cast(T, NT ? __builtin_nontemporal_load(q) : *q);
}

// p: super-block of the tile (wavefront-uniform).
template <int WT, bool NT>
__device__ __forceinline__ uint2 load_q(const uint8_t *p, int b) {
    const unsigned lane = threadIdx.x % kWave, r = lane % 16, kg = lane / 16;
    return load_w<NT, uint2>(p + ((WT == kTypeKQ8 ? 3 : 1) + (kg >> 1)) * 256 + r * 16 + 8 * (kg & 1) + 512 * b);
}
template <int WT, bool MINS, bool NT>
__device__ __forceinline__ void load_h(TileH<WT, MINS> &t, const uint8_t *p) {
    const unsigned o = (threadIdx.x % 16) * 16;
    if constexpr (WT == kTypeKQ8) {
        t.d[0] = load_w<NT, float2>(p + o);
        t.h = load_w<NT, uint4>(p + o + 256);
        if constexpr (MINS) t.m[0] = load_w<NT, uint4>(p + o + 512);
    } else {
        t.h = load_w<NT, uint4>(p + o);
    }
}

// LDS of a work-group: A [CH][K] int8 rows, 16-byte piece p of row t at slot p ^ (t & 15) of its 256-value
// super-block (so the 16 rows a product reads lie in different banks); DX the rows' scales, [K / 32][CH] f32 for Q8_0
// and [K / 256][CH] for Q8_K; BH (Q4_K) the split group sums [K / 256][CH][8]; Z 256 zero bytes (KQ8); the pairs and
// their activation rows.
struct RLds {
    unsigned char *a;
    float *dx;
    unsigned *bh;
    unsigned char *z;
    int *pair, *src;
};

template <int WT>
__host__ __device__ inline size_t r_lds(int CH, int K, unsigned char *base, RLds *o) {
    const size_t a = (size_t) CH * K, dx = (size_t) (WT == kTypeQ8_0 ? K / 32 : K / 256) * CH * 4;
    const size_t bh = WT == kTypeQ4_K ? (size_t) CH * (K / 32) * 4 : 0, z = WT == kTypeKQ8 ? 256 : 0;
    if (o) {
        o->a = base;
        o->z = base + a;
        o->dx = reinterpret_cast<float *>(base + a + z);
        o->bh = reinterpret_cast<unsigned *>(base + a + z + dx);
        o->pair = reinterpret_cast<int *>(base + a + z + dx + bh);
        o->src = o->pair + CH;
    }
    return a + z + dx + bh + (size_t) 2 * CH * 4;
}

// Stages the item's n activation rows. Rows n .. CH - 1 keep stale bytes (their products are never stored), their
// scales repeat row n - 1's.
template <int WT, int CH, int NW>
__device__ __forceinline__ void stage_rows(const GroupedParams &P, const RLds &L, int n) {
    const int tid = threadIdx.x, lane = tid % kWave, wave = __builtin_amdgcn_readfirstlane(tid / kWave);
    const int K = P.K, np = K / 16, nsb = K / 256;
    for (int t = wave; t < n; t += NW) {
        const int8_t *row = P.xqs + (size_t) __builtin_amdgcn_readfirstlane(L.src[t]) * K;
        for (int c0 = 0; c0 < np; c0 += kWave) {
            const int c = c0 + lane;
            if (c < np) __builtin_amdgcn_global_load_lds(row + ((c ^ (t & 15)) * 16), (lds_void *) (L.a + (size_t) t * K + c0 * 16), 16, 0, 0);
        }
    }
    if constexpr (WT == kTypeQ8_0) {
        for (int i = tid; i < CH * (K / 128); i += NW * kWave) {
            const int t = i % CH, q4 = i / CH;
            const float4 v = *reinterpret_cast<const float4 *>(P.xd + (size_t) L.src[min(t, n - 1)] * (K / 32) + 4 * q4);
            L.dx[(4 * q4) * CH + t] = v.x;
            L.dx[(4 * q4 + 1) * CH + t] = v.y;
            L.dx[(4 * q4 + 2) * CH + t] = v.z;
            L.dx[(4 * q4 + 3) * CH + t] = v.w;
        }
    } else {
        for (int i = tid; i < CH * nsb; i += NW * kWave) {
            const int t = i % CH, sb = i / CH;
            L.dx[sb * CH + t] = P.xd[(size_t) L.src[min(t, n - 1)] * (K / 32) + 8 * sb];
        }
    }
    if constexpr (WT == kTypeQ4_K) {
        for (int i = tid; i < CH * nsb * 2; i += NW * kWave) {
            const int t = i % CH, hb = i / CH; // half super-block
            const uint4 v = *reinterpret_cast<const uint4 *>(P.xbh + (size_t) L.src[min(t, n - 1)] * (K / 32) + 4 * hb);
            *reinterpret_cast<uint4 *>(L.bh + ((hb / 2) * CH + t) * 8 + 4 * (hb & 1)) = v;
        }
    }
    if constexpr (WT == kTypeKQ8) {
        if (tid < 64) reinterpret_cast<unsigned *>(L.z)[tid] = 0u;
    }
}

// The activations of block b (0 .. 7) of a super-block for the lane: 8 bytes of row r of every M-tile. KQ8 takes the two 16-value groups apart: lanes kg < 2 hold the first
// (the others zeros), lanes kg >= 2 the second.
template <int WT, int MT>
struct Acts {
    uint2 a[WT == kTypeKQ8 ? 2 : 1][MT];
};
template <int WT, int MT, int CH>
__device__ __forceinline__ void load_acts(Acts<WT, MT> &x, const RLds &L, int K, int sb, int b) {
    const unsigned lane = threadIdx.x % kWave, r = lane % 16, kg = lane / 16;
    // piece 2 b + kg / 2 of row r at slot (2 b + kg / 2) ^ r; b only flips bits 5-7 of the byte offset
    const unsigned a0 = here(r * K + (((kg >> 1) ^ r) * 16) + 8 * (kg & 1)) + sb * 256, zo = (unsigned) (L.z - L.a);
#pragma unroll
    for (int mt = 0; mt < MT; mt++) {
        const unsigned at = a0 + 16 * mt * K;
        if constexpr (WT == kTypeKQ8) {
            x.a[0][mt] = *reinterpret_cast<const uint2 *>(L.a + ((kg < 2 ? at : zo) ^ (b * 32)));
            x.a[1][mt] = *reinterpret_cast<const uint2 *>(L.a + ((kg < 2 ? zo : at) ^ (b * 32)));
        } else {
            x.a[0][mt] = *reinterpret_cast<const uint2 *>(L.a + (at ^ (b * 32)));
        }
    }
}

__device__ __forceinline__ unsigned dw(const uint4 &v, int i) { return i == 0 ? v.x : i == 1 ? v.y : i == 2 ? v.z : v.w; }

// The values as written, here: an empty asm statement (no instruction) that keeps the compiler from delaying or
// regrouping the sums of a block past the next one, which would hold every product of a super-block in registers.
__device__ __forceinline__ void pin(f32x4 &v) {
#pragma unroll
    for (int i = 0; i < 4; i++) asm volatile("" : "+v"(v[i]));
}
__device__ __forceinline__ void pin(i32x4 &v) {
#pragma unroll
    for (int i = 0; i < 4; i++) asm volatile("" : "+v"(v[i]));
}
// Byte `i` of v, sign-extended, as a register of its own (folded into the multiply as a byte select, the product would
// lose the multiply-add form).
__device__ __forceinline__ int sext_byte(unsigned v, int i) {
    int s = (int) (int8_t) (v >> (8 * i));
    asm volatile("" : "+v"(s));
    return s;
}

// Q8_0 rows with an infinite scale (no quantizer writes one): d_w I is +-inf there, but the fma with -1.5 2^23 d_w above
// gives inf - inf. Sums that came out NaN are therefore formed again from plain products, as the GEMV kernels form them
// (and stay NaN where a scale or activation is, or for 0 inf); the others keep their values.
template <int MT, int CH>
__device__ __forceinline__ void rows_plain_q8(const RLds &L, int K, const uint8_t *w0, const uint8_t *w1, f32x4 (&acc)[2][MT]) {
    constexpr int C = chunks_of(kTypeQ8_0);
    const unsigned lane = threadIdx.x % kWave, r = lane % 16, kg = lane / 16;
    f32x4 sum[2][MT];
#pragma unroll
    for (int t = 0; t < 2; t++)
#pragma unroll
        for (int mt = 0; mt < MT; mt++) sum[t][mt] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll 1
    for (int b = 0; b < K / 32; b++) {
        Acts<kTypeQ8_0, MT> x;
        load_acts<kTypeQ8_0, MT, CH>(x, L, K, b / 8, b % 8);
#pragma unroll
        for (int t = 0; t < 2; t++) {
            const uint8_t *w = (t ? w1 : w0) + (size_t) (b / 8) * (C * 256);
            const float d = h2f(*reinterpret_cast<const uint16_t *>(w + r * 16 + 2 * (b % 8)));
            const uint2 q = load_q<kTypeQ8_0, false>(w, b % 8);
#pragma unroll
            for (int mt = 0; mt < MT; mt++) {
                const f32x4 dx = *reinterpret_cast<const f32x4 *>(L.dx + b * CH + 16 * mt + 4 * kg);
                const i32x4 I = mfma8(x.a[0][mt], q, i32x4{0, 0, 0, 0});
#pragma unroll
                for (int i = 0; i < 4; i++) sum[t][mt][i] += (float) I[i] * (d * dx[i]);
            }
        }
    }
#pragma unroll
    for (int t = 0; t < 2; t++)
#pragma unroll
        for (int mt = 0; mt < MT; mt++)
#pragma unroll
            for (int i = 0; i < 4; i++) acc[t][mt][i] = acc[t][mt][i] != acc[t][mt][i] ? sum[t][mt][i] : acc[t][mt][i];
}

// The whole K of the wavefront's two tiles (rows at w0, w1) against the item's rows: acc[tile][mt][i] = token
// 16 mt + 4 (lane / 16) + i of the item, row lane % 16 of the tile. q / h hold super-block 0. A block's quants are
// requested for the next super-block as soon as they have been multiplied, into the same registers, so every load
// has a super-block's products to arrive in and no second copy of the tile is held.
template <int WT, bool MINS, int MT, int CH, bool NT>
__device__ __forceinline__ void rows_products(const RLds &L, int K, const uint8_t *w0, const uint8_t *w1, TileQ<WT> (&q)[2],
                                              TileH<WT, MINS> (&h)[2], f32x4 (&acc)[2][MT]) {
    constexpr int C = chunks_of(WT);
    const unsigned lane = threadIdx.x % kWave, r = lane % 16, kg = lane / 16;
    const int nsb = K / 256;
    const i32x4 zero = {0, 0, 0, 0}, magic = {kMagic, kMagic, kMagic, kMagic};
#pragma unroll
    for (int t = 0; t < 2; t++)
#pragma unroll
        for (int mt = 0; mt < MT; mt++) acc[t][mt] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    const uint8_t *wp[2] = {w0, w1};
    Acts<WT, MT> x;
    load_acts<WT, MT, CH>(x, L, K, 0, 0);
    auto super_block = [&](int sb, auto more_c) __attribute__((always_inline)) {
        constexpr bool more = decltype(more_c)::value;
        TileH<WT, MINS> nh[2]; // (not Q8_0)
#pragma unroll
        for (int t = 0; t < 2; t++) {
            wp[t] += C * 256;
            if constexpr (more && WT != kTypeQ8_0) load_h<WT, MINS, NT>(nh[t], wp[t]);
        }
        i32x4 isum[2][WT == kTypeQ8_0 ? 0 : MT], imin[2][WT == kTypeKQ8 && MINS ? MT : 0];
        f32x4 part[2][WT == kTypeQ8_0 ? MT : 0]; // the super-block's own sum
        unsigned last[2]; // Q8_0: the next super-block's scales of blocks 6 and 7
        unsigned sc[2][2]; // Q4_K: the 6-bit scales, one per byte (sub-blocks 0-3 and 4-7)
        if constexpr (WT != kTypeQ8_0) {
#pragma unroll
            for (int t = 0; t < 2; t++) {
#pragma unroll
                for (int mt = 0; mt < MT; mt++) {
                    isum[t][mt] = zero;
                    if constexpr (WT == kTypeKQ8 && MINS) imin[t][mt] = zero;
                }
                sc[t][0] = h[t].h.y & 0x3f3f3f3fu;
                sc[t][1] = (h[t].h.w & 0x0f0f0f0fu) | ((h[t].h.y >> 2) & 0x30303030u);
            }
        }
#pragma unroll
        for (int b = 0; b < 8; b++) {
            Acts<WT, MT> nx;
            if (b < 7) load_acts<WT, MT, CH>(nx, L, K, sb, b + 1);
            else if constexpr (more) load_acts<WT, MT, CH>(nx, L, K, sb + 1, 0);
            if constexpr (WT == kTypeQ8_0) {
                float d[2], c[2];
                i32x4 I[2][MT];
                f32x4 dx[MT]; // arrive during the products
#pragma unroll
                for (int mt = 0; mt < MT; mt++) dx[mt] = *reinterpret_cast<const f32x4 *>(L.dx + (sb * 8 + b) * CH + 16 * mt + 4 * kg);
#pragma unroll
                for (int t = 0; t < 2; t++) {
                    const unsigned d2 = here(dw(h[t].h, b / 2));
                    d[t] = h2f((b & 1) ? d2 >> 16 : d2);
                    c[t] = -kMagicF * d[t];
#pragma unroll
                    for (int mt = 0; mt < MT; mt++) I[t][mt] = mfma8(x.a[0][mt], q[t].q[b], magic);
                }
#pragma unroll
                for (int mt = 0; mt < MT; mt++)
#pragma unroll
                    for (int t = 0; t < 2; t++)
#pragma unroll
                        for (int i = 0; i < 4; i++) {
                            const float v = fmaf(__int_as_float(I[t][mt][i]), d[t], c[t]);
                            part[t][mt][i] = b == 0 ? dx[mt][i] * v : fmaf(dx[mt][i], v, part[t][mt][i]);
                        }
#pragma unroll
                for (int mt = 0; mt < MT; mt++)
#pragma unroll
                    for (int t = 0; t < 2; t++) pin(part[t][mt]);
            } else if constexpr (WT == kTypeQ4_K) {
                i32x4 I[2][MT];
                int s[2];
#pragma unroll
                for (int t = 0; t < 2; t++) {
                    const uint2 v = q[t].q[b / 2];
                    const uint2 n = (b & 1) ? make_uint2((v.x >> 4) & 0x0f0f0f0fu, (v.y >> 4) & 0x0f0f0f0fu)
                                            : make_uint2(v.x & 0x0f0f0f0fu, v.y & 0x0f0f0f0fu);
                    s[t] = sext_byte(sc[t][b / 4], b % 4);
#pragma unroll
                    for (int mt = 0; mt < MT; mt++) I[t][mt] = mfma8(x.a[0][mt], n, zero);
                }
#pragma unroll
                for (int t = 0; t < 2; t++)
#pragma unroll
                    for (int mt = 0; mt < MT; mt++) {
#pragma unroll
                        for (int i = 0; i < 4; i++) isum[t][mt][i] += __mul24(s[t], I[t][mt][i]);
                        pin(isum[t][mt]);
                    }
            } else {
                int s[2][2];
#pragma unroll
                for (int t = 0; t < 2; t++)
#pragma unroll
                    for (int g = 0; g < 2; g++) s[t][g] = sext_byte(dw(h[t].h, b / 2), (2 * b + g) % 4);
#pragma unroll
                for (int mt = 0; mt < MT; mt++) {
                    i32x4 I[2][2];
#pragma unroll
                    for (int t = 0; t < 2; t++)
#pragma unroll
                        for (int g = 0; g < 2; g++) I[t][g] = mfma8(x.a[g][mt], q[t].q[b], zero);
                    if constexpr (MINS) {
                        const uint2 av = make_uint2(x.a[0][mt].x | x.a[1][mt].x, x.a[0][mt].y | x.a[1][mt].y);
#pragma unroll
                        for (int t = 0; t < 2; t++) {
                            // the lane's 8 values lie in group 2 b + kg / 2
                            const unsigned m = __builtin_amdgcn_perm(0u, dw(h[t].m[0], b / 2), (2 * (b & 1) + (kg >> 1)) * 0x01010101u);
                            imin[t][mt] = mfma8(av, make_uint2(m, m), imin[t][mt]);
                        }
                    }
#pragma unroll
                    for (int t = 0; t < 2; t++)
#pragma unroll
                        for (int g = 0; g < 2; g++) {
#pragma unroll
                            for (int i = 0; i < 4; i++) isum[t][mt][i] += __mul24(s[t][g], I[t][g][i]);
                            pin(isum[t][mt]);
                        }
                }
            }
            if constexpr (more) {
                if (WT != kTypeQ4_K || (b & 1)) {
#pragma unroll
                    for (int t = 0; t < 2; t++) {
                        const int bq = WT == kTypeQ4_K ? b / 2 : b;
                        q[t].q[bq] = load_q<WT, NT>(wp[t], bq);
                    }
                }
                // Q8_0: the scales likewise, in one load once all but the last two blocks' are done (as two halves after blocks 3
                // and 7: 2 VGPRs more, two layers of 512 tokens 407 us instead of 405)
                if (WT == kTypeQ8_0 && b == 5) {
#pragma unroll
                    for (int t = 0; t < 2; t++) {
                        const uint4 v = load_w<NT, uint4>(wp[t] + r * 16);
                        h[t].h.x = v.x, h[t].h.y = v.y, h[t].h.z = v.z;
                        last[t] = v.w;
                    }
                }
                if (WT == kTypeQ8_0 && b == 7) h[0].h.w = last[0], h[1].h.w = last[1];
            }
            if (b < 7 || more) x = nx;
            asm volatile("" ::: "memory"); // the next block's reads stay behind this one's products
            __builtin_amdgcn_sched_barrier(0);
        }
        if constexpr (WT == kTypeQ8_0) {
#pragma unroll
            for (int t = 0; t < 2; t++)
#pragma unroll
                for (int mt = 0; mt < MT; mt++) acc[t][mt] += part[t][mt];
        } else if constexpr (WT == kTypeQ4_K) {
            f32x4 fmin[2][MT];
#pragma unroll
            for (int t = 0; t < 2; t++) {
                const unsigned s1 = h[t].h.z, s2 = h[t].h.w;
                // lanes kg < 2 carry the mins of sub-blocks 4 kg .. 4 kg + 3 as fp16 pairs, the others zeros
                const unsigned mins = (kg == 0 ? s1 & 0x3f3f3f3fu : ((s2 >> 4) & 0x0f0f0f0fu) | ((s1 >> 2) & 0x30303030u)) & (kg < 2 ? ~0u : 0u);
                u32x4 bm;
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    const float mf = (float) ((mins >> (8 * i)) & 0xffu);
                    bm[i] = __builtin_bit_cast(unsigned, __builtin_amdgcn_cvt_pkrtz(mf, mf));
                }
#pragma unroll
                for (int mt = 0; mt < MT; mt++) {
                    const u32x4 bq = *reinterpret_cast<const u32x4 *>(L.bh + (sb * CH + 16 * mt + r) * 8 + 4 * (kg & 1));
                    const f32x4 fz = {0.0f, 0.0f, 0.0f, 0.0f};
                    fmin[t][mt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, bq), __builtin_bit_cast(f16x8, bm), fz, 0, 0, 0);
                }
            }
#pragma unroll
            for (int mt = 0; mt < MT; mt++) {
                const f32x4 dx = *reinterpret_cast<const f32x4 *>(L.dx + sb * CH + 16 * mt + 4 * kg);
#pragma unroll
                for (int t = 0; t < 2; t++) {
                    const float d = h2f(h[t].h.x), dm = h2f(h[t].h.x >> 16);
#pragma unroll
                    for (int i = 0; i < 4; i++)
                        acc[t][mt][i] = fmaf(dx[i], fmaf(d, (float) isum[t][mt][i], -(dm * fmin[t][mt][i])), acc[t][mt][i]);
                }
            }
        } else if constexpr (WT == kTypeKQ8) {
#pragma unroll
            for (int mt = 0; mt < MT; mt++) {
                const f32x4 dx = *reinterpret_cast<const f32x4 *>(L.dx + sb * CH + 16 * mt + 4 * kg);
#pragma unroll
                for (int t = 0; t < 2; t++) {
#pragma unroll
                    for (int i = 0; i < 4; i++) {
                        float v = h[t].d[0].x * (float) isum[t][mt][i];
                        if constexpr (MINS) v = fmaf(-h[t].d[0].y, (float) imin[t][mt][i], v);
                        acc[t][mt][i] = fmaf(dx[i], v, acc[t][mt][i]);
                    }
                }
            }
        }
        if constexpr (more && WT != kTypeQ8_0) {
            h[0] = nh[0];
            h[1] = nh[1];
        }
    };
    for (int sb = 0; sb + 1 < nsb; sb++) super_block(sb, std::true_type{});
    super_block(nsb - 1, std::false_type{});
    if constexpr (WT == kTypeQ8_0) {
        bool nan = false;
#pragma unroll
        for (int t = 0; t < 2; t++)
#pragma unroll
            for (int mt = 0; mt < MT; mt++)
#pragma unroll
                for (int i = 0; i < 4; i++) nan |= acc[t][mt][i] != acc[t][mt][i];
        if (__ballot(nan) != 0ull) rows_plain_q8<MT, CH>(L, K, w0, w1, acc);
    }
}

// Work-group b -> (item, row block): XCD x = b % 8 takes the items [x per, (x + 1) per), all row blocks of an item before
// the next, so an item's activation rows and an expert's weights (its chunks are consecutive items) meet in one L2.
__device__ __forceinline__ bool r_item(const GroupedParams &P, int n_rb, int4 &it, int &rb) {
    const int n_items = *P.n_items, per = (n_items + kRXcds - 1) / kRXcds;
    const int local = blockIdx.x / kRXcds, item = (blockIdx.x % kRXcds) * per + local / n_rb;
    if (local / n_rb >= per || item >= n_items) return false;
    rb = local % n_rb;
    it = P.items[item];
    return true;
}

// DOWN = false: wavefront w computes gate and up of rows 16 (rb NW + w) .. + 15 and stores silu(gate) * up.
// DOWN = true: down rows 32 (rb NW + w) .. + 31, times the pair's router weight.
template <int WT, bool MINS, int MT, bool DOWN, int NW, bool NT>
__global__ __launch_bounds__(NW *kWave, WT == kTypeKQ8 ? (NW == 8 ? 2 : 3) : 4) void rows_kernel(GroupedParams P) {
    constexpr int CH = 16 * MT, C = chunks_of(WT);
    extern __shared__ __align__(16) unsigned char smem[];
    RLds L;
    r_lds<WT>(CH, P.K, smem, &L);
    int4 it;
    int rb;
    if (!r_item(P, P.rows / (DOWN ? 32 * NW : 16 * NW), it, rb)) return;
    const int n = it.z, tid = threadIdx.x, lane = tid % kWave, wave = __builtin_amdgcn_readfirstlane(tid / kWave);
    if (tid < CH) {
        const int p = P.perm[it.y + min(tid, n - 1)];
        L.pair[tid] = p;
        L.src[tid] = p / P.row_div;
    }
    const size_t tb = (size_t) (P.K / 256) * (C * 256); // bytes of a 16-row block
    const int row0 = DOWN ? (rb * NW + wave) * 32 : (rb * NW + wave) * 16;
    const uint8_t *w0 = P.w0 + (size_t) it.x * P.stride0 + (size_t) (row0 / 16) * tb;
    const uint8_t *w1 = DOWN ? w0 + tb : P.w1 + (size_t) it.x * P.stride1 + (size_t) (row0 / 16) * tb;
    __syncthreads();
    stage_rows<WT, CH, NW>(P, L, n);
    TileQ<WT> q[2];
    TileH<WT, MINS> h[2];
    load_h<WT, MINS, NT>(h[0], w0);
    load_h<WT, MINS, NT>(h[1], w1);
#pragma unroll
    for (int b = 0; b < (WT == kTypeQ4_K ? 4 : 8); b++) {
        q[0].q[b] = load_q<WT, NT>(w0, b);
        q[1].q[b] = load_q<WT, NT>(w1, b);
    }
    wait_vm<0>(); // this wavefront's copies into LDS (the weights, requested after them, are needed next anyway)
    __syncthreads();
    const int kg = lane / 16, r = lane % 16;
    f32x4 acc[2][MT];
    rows_products<WT, MINS, MT, CH, NT>(L, P.K, w0, w1, q, h, acc);
#pragma unroll
    for (int mt = 0; mt < MT; mt++) {
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const int pos = 16 * mt + 4 * kg + i;
            if (pos < n) {
                const int p = L.pair[pos];
                float *out = P.out + (size_t) p * P.rows + row0 + r;
                if constexpr (DOWN) {
                    const float wt = P.weights[p];
                    out[0] = acc[0][mt][i] * wt;
                    out[16] = acc[1][mt][i] * wt;
                } else {
                    const float gs = acc[0][mt][i], us = acc[1][mt][i];
                    out[0] = (gs / (1.0f + expf(-gs))) * us;
                }
            }
        }
    }
}

template <int WT, bool MINS, int MT, bool DOWN, int NW, bool NT>
hipError_t launch_rows_n(const GroupedParams &P, int max_items, hipStream_t st, const LaunchTiming *tm) {
    const size_t lds = r_lds<WT>(16 * MT, P.K, nullptr, nullptr);
    static std::atomic<uint64_t> allowed{0};
    const void *kernel = reinterpret_cast<const void *>(&rows_kernel<WT, MINS, MT, DOWN, NW, NT>);
    if (const hipError_t e = allow_dynamic_lds(kernel, 160 * 1024, allowed); e != hipSuccess) return e;
    const int per = (max_items + kRXcds - 1) / kRXcds;
    return launch(rows_kernel<WT, MINS, MT, DOWN, NW, NT>, dim3(kRXcds * per * (P.rows / (DOWN ? 32 * NW : 16 * NW))), dim3(NW * kWave), lds, st, tm, P);
}
// Gate / up work-groups take 8 wavefronts (128 rows) where the staged rows fill 64 KB or more, so that the two
// work-groups a CU holds then are 16 wavefronts: 30B-shaped Q8_0 layer, 32-pair items, us with 4 / 8: 300 Zipf-routed
// tokens 145 / 129, 512 194 / 181, 512 evenly routed 218 / 220; 235B shape, 16-pair Q4_K items, 64 tokens 315 / 295.
// Below that 4 are faster (more work-groups overlap their starts: 64 tokens of Q2_K + Q3_K 159 / 186), and so they are
// for down, whose rows are short (512 tokens Q8_0 214 / 244). (Q8_0 figures from before the super-block sums, which add 1 to 2%
// to either side.)
template <int WT, bool MINS, int MT, bool DOWN, bool NT>
hipError_t launch_rows_w(const GroupedParams &P, int max_items, hipStream_t st, const LaunchTiming *tm) {
    if constexpr (!DOWN)
        if (16 * MT * P.K >= 64 * 1024 && P.rows % 128 == 0) return launch_rows_n<WT, MINS, MT, false, 8, NT>(P, max_items, st, tm);
    return launch_rows_n<WT, MINS, MT, DOWN, 4, NT>(P, max_items, st, tm);
}
template <int WT, bool MINS, int MT, bool DOWN>
hipError_t launch_rows_t(const GroupedParams &P, int max_items, hipStream_t st, const LaunchTiming *tm) {
    if constexpr (MT == 1)
        if (P.once) return launch_rows_w<WT, MINS, MT, DOWN, true>(P, max_items, st, tm);
    return launch_rows_w<WT, MINS, MT, DOWN, false>(P, max_items, st, tm);
}

template <bool DOWN>
hipError_t launch_rows(const GroupedParams &P, int max_items, hipStream_t st, const LaunchTiming *tm) {
    if (max_items <= 0) return hipSuccess;
    if ((P.chunk != 16 && (P.chunk != 32 || P.type != kTypeQ8_0)) || P.K % 256 != 0 || P.rows % (DOWN ? 128 : 64) != 0) return hipErrorInvalidValue;
    switch (P.type) {
        case kTypeQ8_0:
            return P.chunk == 16 ? launch_rows_t<kTypeQ8_0, false, 1, DOWN>(P, max_items, st, tm)
                                 : launch_rows_t<kTypeQ8_0, false, 2, DOWN>(P, max_items, st, tm);
        case kTypeQ4_K: return P.xbh ? launch_rows_t<kTypeQ4_K, true, 1, DOWN>(P, max_items, st, tm) : hipErrorInvalidValue;
        case kTypeQ2_K:
        case kTypeQ5_K: return launch_rows_t<kTypeKQ8, true, 1, DOWN>(P, max_items, st, tm);
        default: return launch_rows_t<kTypeKQ8, false, 1, DOWN>(P, max_items, st, tm); // Q3_K and Q6_K have no mins
    }
}

}  // namespace

hipError_t launch_gate_up_rows(const GroupedParams &P, int max_items, hipStream_t st, const LaunchTiming *tm) {
    return launch_rows<false>(P, max_items, st, tm);
}

hipError_t launch_down_rows(const GroupedParams &P, int max_items, hipStream_t st, const LaunchTiming *tm) {
    return launch_rows<true>(P, max_items, st, tm);
}

}  // namespace lstk
