// pk_tile.h - the wide matrix-core tile: 32 weight rows per wave times up to
// 128 q8_K rows per block, on v_mfma_i32_16x16x64_i8.
//
// What bounds a prompt chunk is not its bytes but the work per product: the
// 16-row tiles of mmq.hip scale every 32-value sum in the vector unit (4
// multiply-adds per lane and MFMA) and stage raw weights through LDS for
// every 32 tokens. Here the integer scales go into the weights instead: a
// wave decodes its 32 rows of a super-block once, in registers, into int8
// operands that already carry their sub-block scale, so the MFMAs of a
// super-block chain without any vector work between them, and one fp32 step
// per (row, token, super-block) is left. A product code * scale that does not
// fit int8 is split in two digits, lo + 2^kShift * hi, each an int8 operand
// of its own (two MFMAs, still exact int32 sums).
//
// Operands (lane l: i = l & 15, q = l >> 4): A[i][k] token i, B[k][j] weight
// row j, 16 int8 of lane group q each; D[i][j]: lane j + 16 (i / 4), element
// i % 4. A lane decodes rows i (tile 0) and 16 + i (tile 1) itself, so their
// scales are scalars of the lane. A super-block is 4 steps of 64 values; the
// 16 values a lane group holds in a step are piece F::piece(s, q) of the
// super-block (16 values each), chosen so that each lane loads every code
// byte of its share once. The min terms sum_c bsums[c] * min_c run as one
// v_mfma_f32_16x16x16_f16 (lane group q: bsums 4q .. 4q + 3): a q8_K bsum
// (|.| <= 2048) and a min (<= 63) are exact in f16 and every partial sum is
// below 2^24, so the fp32 result is the exact integer.
#pragma once

#include <type_traits>

#include "pk_rowdot.h"

namespace pk {

typedef int32_t v4i_t __attribute__((ext_vector_type(4)));
typedef float v4f_t __attribute__((ext_vector_type(4)));
typedef _Float16 v4h_t __attribute__((ext_vector_type(4)));
typedef _Float16 v2h_t __attribute__((ext_vector_type(2)));
typedef unsigned short v2u16_t __attribute__((ext_vector_type(2)));

PK_DEV v4i_t mfma64(uint4 a, uint4 b, v4i_t c) {
    return __builtin_amdgcn_mfma_i32_16x16x64_i8(__builtin_bit_cast(v4i_t, a), __builtin_bit_cast(v4i_t, b), c, 0, 0,
                                                 0);
}
PK_DEV v4f_t mfma16_f16(uint2 a, uint2 b) {
    const v4f_t z = {};
    return __builtin_amdgcn_mfma_f32_16x16x16f16(__builtin_bit_cast(v4h_t, a), __builtin_bit_cast(v4h_t, b), z, 0, 0,
                                                 0);
}

// Per 16-bit half, modulo 2^16: a * b and a * b + c
PK_DEV uint32_t half_mul(uint32_t a, uint32_t b) {
    return __builtin_bit_cast(uint32_t, __builtin_bit_cast(v2u16_t, a) * __builtin_bit_cast(v2u16_t, b));
}
PK_DEV uint32_t half_mad(uint32_t a, uint32_t b, uint32_t c) {
    return __builtin_bit_cast(uint32_t, __builtin_bit_cast(v2u16_t, a) * __builtin_bit_cast(v2u16_t, b) +
                                                __builtin_bit_cast(v2u16_t, c));
}
PK_DEV uint32_t dup16(uint32_t v) { return __builtin_amdgcn_perm(v, v, 0x01000100u); }
// byte b of w in the low byte of both halves, the high bytes 0
PK_DEV uint32_t dup_byte(uint32_t w, uint32_t b) { return __builtin_amdgcn_perm(0u, w, 0x0C000C00u + b * 0x00010001u); }
PK_DEV uint32_t word4(uint4 v, uint32_t i) { return i == 0 ? v.x : i == 1 ? v.y : i == 2 ? v.z : v.w; }

// f16 pair (bytes b0, b1 of w, integers 0..255): 0x6400 | byte is 1024 + byte
PK_DEV uint32_t f16_of_bytes(uint32_t w, uint32_t b0, uint32_t b1) {
    const uint32_t v = __builtin_amdgcn_perm(0x64646464u, w, 0x04000400u + b0 + (b1 << 16));
    const v2h_t off = {(_Float16)-1024.0f, (_Float16)-1024.0f};
    return __builtin_bit_cast(uint32_t, __builtin_bit_cast(v2h_t, v) + off);
}
// f16 pair of two int16
PK_DEV uint32_t f16_of_i16(uint32_t w) {
    const v2h_t v = {(_Float16)(int16_t)(w & 0xffffu), (_Float16)(int16_t)(w >> 16)};
    return __builtin_bit_cast(uint32_t, v);
}

// Four unsigned codes u (bytes) times a signed scale, p = (u - bias) * s with
// |p| < 2^15 - 128, split p = lo + 256 hi: in 16-bit halves p + 128 = u * s +
// (128 - bias * s), whose high byte is hi and whose low byte is lo + 128.
PK_DEV void split_product(uint32_t u, uint32_t s2, uint32_t k2, uint32_t &lo, uint32_t &hi) {
    const uint32_t e = half_mad(u & 0x00ff00ffu, s2, k2), o = half_mad((u >> 8) & 0x00ff00ffu, s2, k2);
    lo = __builtin_amdgcn_perm(o, e, 0x06020400u) ^ 0x80808080u;
    hi = __builtin_amdgcn_perm(o, e, 0x07030501u);
}

// One row's decoded super-block: the lo (and hi) operands of the 4 steps,
// the f16 mins of lane group q's bsums, xd and xmin.
struct TileW {
    uint4 lo[4], hi[4];
    uint2 mins;
    float xd, xmin;
};

template <uint32_t Q>
struct TileFmt;

// The words of a Raw as values the compiler must have in registers here: its
// loads cannot be moved past this point, to where the words are decoded.
template <typename Raw>
PK_DEV void hold_raw(Raw &r) {
    struct Words {
        uint32_t v[sizeof(Raw) / 4u];
    } w = __builtin_bit_cast(Words, r);
#pragma unroll
    for (uint32_t k = 0; k < sizeof(Raw) / 4u; k++) asm volatile("" : "+v"(w.v[k]));
    r = __builtin_bit_cast(Raw, w);
}

// the 6-bit scales and mins of the Q4_K / Q5_K header (cpu_dot.rs:147-156), a
// byte each
struct KqScales {
    uint32_t sc0, sc1, mn0, mn1;  // sub-blocks 0..3, 4..7
};
PK_DEV KqScales kq_scales(uint4 hdr) {
    KqScales k;
    k.sc0 = hdr.y & 0x3f3f3f3fu;
    k.mn0 = hdr.z & 0x3f3f3f3fu;
    k.sc1 = (hdr.w & 0x0f0f0f0fu) | ((hdr.y >> 2) & 0x30303030u);
    k.mn1 = ((hdr.w >> 4) & 0x0f0f0f0fu) | ((hdr.z >> 2) & 0x30303030u);
    return k;
}
// bsums 4q + j carry min (4q + j) / 2 = 2q + j / 2: bytes 2 (q % 2), + 1 of
// word q / 2
PK_DEV uint2 kq_mins(const KqScales &k, uint32_t q) {
    const uint32_t m = (q & 2u ? k.mn1 : k.mn0) >> (16u * (q & 1u));
    return make_uint2(f16_of_bytes(m, 0, 0), f16_of_bytes(m, 1, 1));
}

// Q4_K: lane group q holds 16-byte pieces q and q + 4 of qs, low nibbles in
// steps 0 and 2, high in 1 and 3: sub-block 4 (s / 2) + 2 (q / 2) + s % 2.
// Codes 0..15, scale 8 sh + sl with sl, sh < 8: code * digit <= 105, so one
// 16-bit multiply scales two code bytes without a carry between them.
template <>
struct TileFmt<PULSAR_QUANT_Q4_K> {
    static constexpr uint32_t kSb = 144, kShift = 3;
    static constexpr bool kHi = true, kMin = true, kNeg = false;
    struct Raw {
        uint4 q[2], hdr;
    };
    PK_DEV static uint32_t piece(uint32_t s, uint32_t q) { return 8u * (s >> 1) + 2u * (s & 1u) + 4u * (q >> 1) + (q & 1u); }
    PK_DEV static Raw load(const uint8_t *b, uint32_t q) {
        Raw r;
        r.hdr = ldw128(b);
        r.q[0] = ldw128(b + 16u + 16u * q);
        r.q[1] = ldw128(b + 80u + 16u * q);
        return r;
    }
    PK_DEV static void decode(const Raw &r, uint32_t q, const uint2 *, TileW &w) {
        const KqScales k = kq_scales(r.hdr);
        w.mins = kq_mins(k, q);
        w.xd = f16f((uint16_t)r.hdr.x);
        w.xmin = f16f((uint16_t)(r.hdr.x >> 16));
#pragma unroll
        for (uint32_t s = 0; s < 4; s++) {
            const uint32_t v = (s >> 1 ? k.sc1 : k.sc0) >> (16u * (q >> 1));
            const uint32_t sl = dup_byte(v & 0x0707u, s & 1u), sh = dup_byte((v >> 3) & 0x0707u, s & 1u);
            const uint4 x = r.q[s >> 1];
            const uint32_t n = 4u * (s & 1u), m = 0x0f0f0f0fu;
            const uint4 c = make_uint4((x.x >> n) & m, (x.y >> n) & m, (x.z >> n) & m, (x.w >> n) & m);
            w.lo[s] = make_uint4(half_mul(c.x, sl), half_mul(c.y, sl), half_mul(c.z, sl), half_mul(c.w, sl));
            w.hi[s] = make_uint4(half_mul(c.x, sh), half_mul(c.y, sh), half_mul(c.z, sh), half_mul(c.w, sh));
        }
    }
};

// Q5_K: Q4_K's pieces, codes 0..31 (the fifth bit: the sub-block's bit of qh
// byte 16 (q % 2) + i), product split.
template <>
struct TileFmt<PULSAR_QUANT_Q5_K> {
    static constexpr uint32_t kSb = 176, kShift = 8;
    static constexpr bool kHi = true, kMin = true, kNeg = false;
    struct Raw {
        uint4 q[2], hdr, qh;
    };
    PK_DEV static uint32_t piece(uint32_t s, uint32_t q) { return TileFmt<PULSAR_QUANT_Q4_K>::piece(s, q); }
    PK_DEV static Raw load(const uint8_t *b, uint32_t q) {
        Raw r;
        r.hdr = ldw128(b);
        r.qh = ldw128(b + 16u + 16u * (q & 1u));
        r.q[0] = ldw128(b + 48u + 16u * q);
        r.q[1] = ldw128(b + 112u + 16u * q);
        return r;
    }
    PK_DEV static void decode(const Raw &r, uint32_t q, const uint2 *, TileW &w) {
        const KqScales k = kq_scales(r.hdr);
        w.mins = kq_mins(k, q);
        w.xd = f16f((uint16_t)r.hdr.x);
        w.xmin = f16f((uint16_t)(r.hdr.x >> 16));
        const uint32_t hs = 2u * (q >> 1);
        const uint4 qh = make_uint4(r.qh.x >> hs, r.qh.y >> hs, r.qh.z >> hs, r.qh.w >> hs);
#pragma unroll
        for (uint32_t s = 0; s < 4; s++) {
            const uint32_t s2 = dup_byte((s >> 1 ? k.sc1 : k.sc0) >> (16u * (q >> 1)), s & 1u);
            const uint4 x = r.q[s >> 1];
            auto u = [&](uint32_t c, uint32_t h) {
                return ((c >> (4u * (s & 1u))) & 0x0f0f0f0fu) | (((h >> (4u * (s >> 1) + (s & 1u))) & 0x01010101u) << 4);
            };
            split_product(u(x.x, qh.x), s2, 0x00800080u, w.lo[s].x, w.hi[s].x);
            split_product(u(x.y, qh.y), s2, 0x00800080u, w.lo[s].y, w.hi[s].y);
            split_product(u(x.z, qh.z), s2, 0x00800080u, w.lo[s].z, w.hi[s].z);
            split_product(u(x.w, qh.w), s2, 0x00800080u, w.lo[s].w, w.hi[s].w);
        }
    }
};

// Q6_K: lane group q holds 16-byte pieces q and q + 4 of ql (halves h = 0, 1
// of the super-block), low nibbles (quarter q / 2) in steps 2h, high (quarter
// 2 + q / 2) in 2h + 1; scale 4s + q. Codes 0..63 less 32 times a signed
// byte, product split (|p| <= 4096).
template <>
struct TileFmt<PULSAR_QUANT_Q6_K> {
    static constexpr uint32_t kSb = 210, kShift = 8;
    static constexpr bool kHi = true, kMin = false, kNeg = false;
    struct Raw {
        uint4 ql[2], qh, sc;
        uint32_t d;
    };
    PK_DEV static uint32_t piece(uint32_t s, uint32_t q) { return 4u * s + q; }
    PK_DEV static Raw load(const uint8_t *b, uint32_t q) {
        Raw r;
        r.ql[0] = ldw128(b + 16u * q);
        r.ql[1] = ldw128(b + 64u + 16u * q);
        r.qh = ldw128(b + 128u + 16u * q);
        r.sc = ldw128(b + 192u);
        r.d = ldw16(b + 208u);
        return r;
    }
    PK_DEV static void decode(const Raw &r, uint32_t q, const uint2 *, TileW &w) {
        w.xd = f16f((uint16_t)r.d);
        w.xmin = 0.0f;
        const uint32_t hs = 2u * (q >> 1);
        // lane group q loaded qh piece q (half q / 2, bytes 16 (q % 2)); it
        // needs the pieces q % 2 and 2 + q % 2, its own and lane group q ^ 2's
        uint32_t qx[2][4];
#pragma unroll
        for (uint32_t k = 0; k < 4; k++) {
            const auto v = __builtin_amdgcn_permlane32_swap(word4(r.qh, k), word4(r.qh, k), false, false);
            qx[0][k] = v[0];
            qx[1][k] = v[1];
        }
#pragma unroll
        for (uint32_t s = 0; s < 4; s++) {
            const uint32_t s2 = dup16((uint32_t)(int32_t)(int8_t)(word4(r.sc, s) >> (8u * q)));
            const uint32_t k2 = half_mad(s2, 0xffe0ffe0u, 0x00800080u);  // 128 - 32 sc
            const uint4 l = r.ql[s >> 1];
            const uint4 qh = make_uint4(qx[s >> 1][0], qx[s >> 1][1], qx[s >> 1][2], qx[s >> 1][3]);
            auto u = [&](uint32_t c, uint32_t h) {
                return ((c >> (4u * (s & 1u))) & 0x0f0f0f0fu) | (((h >> (hs + 4u * (s & 1u))) & 0x03030303u) << 4);
            };
            split_product(u(l.x, qh.x), s2, k2, w.lo[s].x, w.hi[s].x);
            split_product(u(l.y, qh.y), s2, k2, w.lo[s].y, w.hi[s].y);
            split_product(u(l.z, qh.z), s2, k2, w.lo[s].z, w.hi[s].z);
            split_product(u(l.w, qh.w), s2, k2, w.lo[s].w, w.hi[s].w);
        }
    }
};

// Q2_K: lane group q holds 16-byte piece q of qs, bits 2s, 2s + 1 in step s
// (values 128 (q / 2) + 32 s + 16 (q % 2)); codes 0..3 times a 4-bit scale
// (<= 45), one operand.
template <>
struct TileFmt<PULSAR_QUANT_Q2_K> {
    static constexpr uint32_t kSb = 84, kShift = 0;
    static constexpr bool kHi = false, kMin = true, kNeg = false;
    struct Raw {
        uint4 q;
        uint2 sc;  // scale bytes 8 (q / 2) + [0, 8)
        uint32_t dd;
    };
    PK_DEV static uint32_t piece(uint32_t s, uint32_t q) { return 8u * (q >> 1) + 2u * s + (q & 1u); }
    PK_DEV static Raw load(const uint8_t *b, uint32_t q) {
        Raw r;
        r.sc = ldw64(b + 8u * (q >> 1));
        r.q = ldw128(b + 16u + 16u * q);
        r.dd = ldw32(b + 80u);
        return r;
    }
    PK_DEV static void decode(const Raw &r, uint32_t q, const uint2 *, TileW &w) {
        w.xd = f16f((uint16_t)r.dd);
        w.xmin = f16f((uint16_t)(r.dd >> 16));
        const uint32_t m = ((q & 1u ? r.sc.y : r.sc.x) >> 4) & 0x0f0f0f0fu;  // mins 4q + [0, 4)
        w.mins = make_uint2(f16_of_bytes(m, 0, 1), f16_of_bytes(m, 2, 3));
#pragma unroll
        for (uint32_t s = 0; s < 4; s++) {
            const uint32_t s2 = dup_byte(((s >> 1 ? r.sc.y : r.sc.x) >> (8u * (q & 1u))) & 0x0f0f0f0fu, 2u * (s & 1u));
            const uint32_t n = 2u * s, c = 0x03030303u;
            w.lo[s] = make_uint4(half_mul((r.q.x >> n) & c, s2), half_mul((r.q.y >> n) & c, s2),
                                 half_mul((r.q.z >> n) & c, s2), half_mul((r.q.w >> n) & c, s2));
        }
    }
};

// Q3_K (110 B: hmask[32], qs[64], scales[12], f16 d): Q2_K's pieces and scale
// order. (u - 4) * s with u the 3-bit code and s in [-32, 31] is in [-124,
// 128], so its negative fits int8: one operand, the sum negated (kNeg). Two
// codes per 16-bit half: u * -s + (4 s + 128) is in [0, 252] for each byte,
// so no carry crosses, and xor 0x80 takes the 128 off again.
template <>
struct TileFmt<PULSAR_QUANT_Q3_K> {
    static constexpr uint32_t kSb = 110, kShift = 0;
    static constexpr bool kHi = false, kMin = false, kNeg = true;
    struct Raw {
        uint4 q, hm, tail;  // tail: bytes 94..109 (qs[62..63], scales, d)
    };
    PK_DEV static uint32_t piece(uint32_t s, uint32_t q) { return TileFmt<PULSAR_QUANT_Q2_K>::piece(s, q); }
    PK_DEV static Raw load(const uint8_t *b, uint32_t q) {
        Raw r;
        r.hm = ldw128(b + 16u * (q & 1u));
        r.q = ldw128(b + 32u + 16u * q);
        r.tail = ldw128(b + 94u);
        return r;
    }
    PK_DEV static void decode(const Raw &r, uint32_t q, const uint2 *, TileW &w) {
        w.xd = f16f((uint16_t)(r.tail.w >> 16));
        w.xmin = 0.0f;
        // scale bytes s[0..3], s[4..7], s[8..11]
        const uint32_t s0 = __builtin_amdgcn_alignbyte(r.tail.y, r.tail.x, 2u);
        const uint32_t s1 = __builtin_amdgcn_alignbyte(r.tail.z, r.tail.y, 2u);
        const uint32_t s2 = __builtin_amdgcn_alignbyte(r.tail.w, r.tail.z, 2u);
        // 6-bit scales 8 (q / 2) + 4v + b (cpu_dot.rs:133-145): low bits byte b
        // of s0 / s1 (high nibbles for the upper 8), high bits byte b of s2
        const uint32_t ls = 4u * (q >> 1), lo4 = 0x0f0f0f0fu, hi2 = 0x30303030u;
        const uint32_t h4 = q & 2u ? s2 : s2 << 4;  // bits 2v + 4 (q / 2) to 4 + 2v
        const uint32_t sw[2] = {((s0 >> ls) & lo4) | (h4 & hi2), ((s1 >> ls) & lo4) | ((h4 >> 2) & hi2)};
        const uint32_t hs = 4u * (q >> 1);
        const uint4 hm = make_uint4(r.hm.x >> hs, r.hm.y >> hs, r.hm.z >> hs, r.hm.w >> hs);
#pragma unroll
        for (uint32_t s = 0; s < 4; s++) {
            const uint32_t sc = dup_byte(sw[s >> 1] >> (8u * (q & 1u)), 2u * (s & 1u));
            const uint32_t neg = half_mad(sc, 0xffffffffu, 0x00200020u);  // 32 - sc = -s
            const uint32_t k2 = half_mul(sc, 0x04040404u);                // (4 s + 128) * 257 with s = sc - 32
            const uint32_t n = 2u * s;
            auto one = [&](uint32_t c, uint32_t h) {
                const uint32_t u = ((c >> n) & 0x03030303u) | (((h >> s) & 0x01010101u) << 2);
                return half_mad(u, neg, k2) ^ 0x80808080u;
            };
            w.lo[s] = make_uint4(one(r.q.x, hm.x), one(r.q.y, hm.y), one(r.q.z, hm.z), one(r.q.w, hm.w));
        }
    }
};

// IQ4_XS (136 B: f16 d, u16 scales_h, scales_l[4], qs[128]): lane group q
// holds blocks q and q + 4 of 32, low nibbles in steps 0 and 2, high in 1 and
// 3. The codebook value plus 128 (unsigned) times the 6-bit scale less 32,
// product split.
template <>
struct TileFmt<PULSAR_QUANT_IQ4_XS> {
    static constexpr uint32_t kSb = 136, kShift = 8;
    static constexpr bool kHi = true, kMin = false, kNeg = false;
    struct Raw {
        uint4 q[2];
        uint2 hdr;
    };
    PK_DEV static uint32_t piece(uint32_t s, uint32_t q) { return 8u * (s >> 1) + 2u * q + (s & 1u); }
    PK_DEV static Raw load(const uint8_t *b, uint32_t q) {
        Raw r;
        r.hdr = ldw64(b);
        r.q[0] = ldw128(b + 8u + 16u * q);
        r.q[1] = ldw128(b + 72u + 16u * q);
        return r;
    }
    PK_DEV static void decode(const Raw &r, uint32_t q, const uint2 *, TileW &w) {
        w.xd = f16f((uint16_t)r.hdr.x);
        w.xmin = 0.0f;
        const uint32_t sl = r.hdr.y >> (4u * q), sh = r.hdr.x >> (16u + 2u * q);
#pragma unroll
        for (uint32_t s = 0; s < 4; s++) {
            const uint32_t k = s >> 1;
            const int32_t sc = (int32_t)(((sl >> (16u * k)) & 0x0fu) | (((sh >> (8u * k)) & 3u) << 4)) - 32;
            const uint32_t s2 = dup16((uint32_t)sc);
            const uint32_t k2 = half_mad(s2, 0xff80ff80u, 0x00800080u);  // 128 - 128 sc
            const uint32_t n = 4u * (s & 1u);
            auto u = [&](uint32_t c) { return iq4nl_kv4(c >> n) ^ 0x80808080u; };
            split_product(u(r.q[k].x), s2, k2, w.lo[s].x, w.hi[s].x);
            split_product(u(r.q[k].y), s2, k2, w.lo[s].y, w.hi[s].y);
            split_product(u(r.q[k].z), s2, k2, w.lo[s].z, w.hi[s].z);
            split_product(u(r.q[k].w), s2, k2, w.lo[s].w, w.hi[s].w);
        }
    }
};

// IQ2_XXS (66 B: f16 d, 8 x {aux0, aux1}): lane group q holds grid entries
// 2 (q % 2), + 1 of group 2s + q / 2 in step s; signed magnitudes (<= 43) plus
// 64 times the odd scale 2 ls + 1 (<= 31), product split. Value 0.125 d * sum.
template <>
struct TileFmt<PULSAR_QUANT_IQ2_XXS> {
    static constexpr uint32_t kSb = 66, kShift = 8;
    static constexpr bool kHi = true, kMin = false, kNeg = false;
    struct Raw {
        uint2 a[4];
        uint32_t d;
    };
    PK_DEV static uint32_t piece(uint32_t s, uint32_t q) { return 4u * s + q; }
    PK_DEV static Raw load(const uint8_t *b, uint32_t q) {
        Raw r;
        r.d = ldw16(b);
#pragma unroll
        for (uint32_t s = 0; s < 4; s++) r.a[s] = ldw64(b + 2u + 16u * s + 8u * (q >> 1));
        return r;
    }
    PK_DEV static void decode(const Raw &r, uint32_t q, const uint2 *lut, TileW &w) {
        w.xd = 0.125f * f16f((uint16_t)r.d);
        w.xmin = 0.0f;
#pragma unroll
        for (uint32_t s = 0; s < 4; s++) {
            const uint2 a = r.a[s];
            const uint32_t s2 = dup16(2u * (a.y >> 28) + 1u);
            const uint32_t k2 = half_mad(s2, 0xffc0ffc0u, 0x00800080u);  // 128 - 64 sc
            const uint32_t ix = a.x >> (16u * (q & 1u)), sg = a.y >> (14u * (q & 1u));
            uint32_t v[4];
            iq2_signed8(lut, ix & 0xffu, sg & 127u, v[0], v[1]);
            iq2_signed8(lut, (ix >> 8) & 0xffu, (sg >> 7) & 127u, v[2], v[3]);
            // v + 64 per byte: v in [-43, 43], so no byte borrows
            split_product((v[0] ^ 0x80808080u) - 0x40404040u, s2, k2, w.lo[s].x, w.hi[s].x);
            split_product((v[1] ^ 0x80808080u) - 0x40404040u, s2, k2, w.lo[s].y, w.hi[s].y);
            split_product((v[2] ^ 0x80808080u) - 0x40404040u, s2, k2, w.lo[s].z, w.hi[s].z);
            split_product((v[3] ^ 0x80808080u) - 0x40404040u, s2, k2, w.lo[s].w, w.hi[s].w);
        }
    }
};

// A block of 4 waves: WR groups of 32 weight rows x WK slices of K (WR WK =
// 4), NS slices of 16 tokens. An iteration takes WK super-blocks, wave (wr,
// wk) super-block wk of them; the WK partial sums are added in slice order at
// the end. The tokens' q8_K records (token t, super-block k of the iteration:
// record k kTok + t) are copied to LDS by the memory pipeline itself
// (global_load_lds, no registers), one iteration ahead, into the other of two
// buffers; the weights go straight to the registers of the wave that decodes
// them, also one iteration ahead. Within a wave the fp32 step of a token
// slice is issued between the MFMAs of the next one.
template <uint32_t Q, uint32_t WR, uint32_t WK, uint32_t NS>
struct Tile {
    using F = TileFmt<Q>;
    static_assert(WR * WK == 4, "4 waves");
    static constexpr uint32_t kTok = 16u * NS, kRec = WK * kTok;
    // A buffer: 256 q8 bytes per record, then 32 bytes of bsums (formats with
    // mins), then the records' d. A DMA instruction writes 64 consecutive 16-
    // byte slots, so the records cannot be padded apart; piece p of record r
    // sits in slot p ^ (r % 16) of the record instead, which puts the pieces
    // that 16 lanes read together on distinct banks.
    static constexpr uint32_t kBsum = kRec * 256u, kD = kBsum + (F::kMin ? kRec * 32u : 0u);
    static constexpr uint32_t kBuf = kD + kRec * 4u;
    static_assert(kRec % 64u == 0, "whole DMA instructions");

    float acc[NS][2][4];  // [slice][row tile][token 4q + r]

    // w0, w1: the lane's two weight rows; xb + off_of(t): the q8_K row of token
    // t < np (0 < np <= kTok); buf0, buf1: kBuf bytes each, two distinct LDS
    // arrays. On return the lanes
    // of wave (wr, wk) hold the sums of their share of the elements (mine()).
    template <typename OffOf>
    PK_DEV void run(uint8_t *buf0, uint8_t *buf1, const uint2 *lut, const uint8_t *w0, const uint8_t *w1, uint32_t nb,
                    uint32_t np, const uint8_t *xb, OffOf off_of) {
        const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
        const uint32_t i = lane & 15u, q = lane >> 4, wk = wave / WR;
        auto clamp_sb = [&](uint32_t sb) { return (sb < nb ? sb : nb - 1u); };
        // byte `at` of record rec of iteration it (tokens past np: the last one again)
        auto src = [&](uint32_t it, uint32_t rec, uint32_t at) {
            const uint32_t t = rec % kTok;
            const auto o = off_of(t < np ? t : np - 1u) + at;
            if constexpr (WK == 1u)
                return (const PK_GLOBAL uint32_t *)(xb + clamp_sb(it) * 292u + o);
            else
                return (const PK_GLOBAL uint32_t *)(xb + (o + clamp_sb(it * WK + rec / kTok) * 292u));
        };
        // every wave issues the same number of instructions; where there are
        // fewer than waves, some write the same bytes twice
        auto dma = [&](uint8_t *buf, uint32_t it) {
#pragma unroll
            for (uint32_t m = 0; m < kRec / 16u; m++) {
                const uint32_t r0 = 4u * (wave + 4u * m), rec = r0 + lane / 16u;
                __builtin_amdgcn_global_load_lds(src(it, rec, 4u + 16u * ((lane ^ rec) & 15u)),
                                                 (PK_LDS uint32_t *)(buf + r0 * 256u), 16, 0, 0);
            }
            if (F::kMin) {
                const uint32_t b = kRec >= 128u ? wave : wave % (kRec / 32u);
                __builtin_amdgcn_global_load_lds(src(it, 32u * b + lane / 2u, 260u + 16u * (lane & 1u)),
                                                 (PK_LDS uint32_t *)(buf + kBsum + 1024u * b), 16, 0, 0);
            }
            const uint32_t y = wave % (kRec / 64u);
            __builtin_amdgcn_global_load_lds(src(it, 64u * y + lane, 0u), (PK_LDS uint32_t *)(buf + kD + 256u * y), 4, 0, 0);
        };
#pragma unroll
        for (uint32_t n = 0; n < NS; n++)
#pragma unroll
            for (int r = 0; r < 4; r++) acc[n][0][r] = acc[n][1][r] = 0.0f;
        // byte offset of the lane's piece of step s within a buffer (token
        // slice 0 of its K slice)
        uint32_t ao[4];
#pragma unroll
        for (uint32_t s = 0; s < 4; s++) ao[s] = (wk * kTok + i) * 256u + 16u * (F::piece(s, q) ^ i);
        const uint32_t n_it = (nb + WK - 1u) / WK;
        dma(buf0, 0u);
        typename F::Raw raw[2];
        auto load_w = [&](uint32_t it) {  // past the end: the last super-block again
            const uint64_t o = (uint64_t)clamp_sb(it * WK + wk) * F::kSb;
            raw[0] = F::load(w0 + o, q);
            raw[1] = F::load(w1 + o, q);
        };
        load_w(0u);
        auto arrived = [] {
            __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0): the wave's DMA writes are in LDS
            __syncthreads();
        };
        auto step = [&](const uint8_t *buf, uint8_t *nbuf, uint32_t it) {
            const bool live = WK == 1u || it * WK + wk < nb;  // wave-uniform
            TileW tw[2];
            F::decode(raw[0], q, lut, tw[0]);
            F::decode(raw[1], q, lut, tw[1]);
            __builtin_amdgcn_sched_barrier(0);
            dma(nbuf, it + 1u);
            load_w(it + 1u);
            uint4 a[2][4];
            auto read_a = [&](uint32_t n) {
#pragma unroll
                for (uint32_t s = 0; s < 4; s++) a[n & 1u][s] = *(const uint4 *)(buf + ao[s] + 4096u * n);
            };
            // the fp32 step of slice n from its sums
            auto finish = [&](uint32_t n, const v4i_t (&dl)[2], const v4i_t (&dh)[2]) {
                const uint4 y4 = *(const uint4 *)(buf + kD + (wk * kTok + 16u * n + 4u * q) * 4u);
                const float yd[4] = {__uint_as_float(y4.x), __uint_as_float(y4.y), __uint_as_float(y4.z),
                                     __uint_as_float(y4.w)};
                v4f_t ms[2];
                if constexpr (F::kMin) {
                    const uint2 b = *(const uint2 *)(buf + kBsum + (wk * kTok + 16u * n + i) * 32u + 8u * q);
                    const uint2 bh = make_uint2(f16_of_i16(b.x), f16_of_i16(b.y));
                    ms[0] = mfma16_f16(bh, tw[0].mins);
                    ms[1] = mfma16_f16(bh, tw[1].mins);
                }
#pragma unroll
                for (int rt = 0; rt < 2; rt++)
#pragma unroll
                    for (int r = 0; r < 4; r++) {
                        const int32_t sum = F::kHi ? (int32_t)((uint32_t)dh[rt][r] << F::kShift) + dl[rt][r] : dl[rt][r];
                        float v = (F::kNeg ? -tw[rt].xd : tw[rt].xd) * (float)sum;
                        if (F::kMin) v = __builtin_fmaf(-tw[rt].xmin, ms[rt][r], v);
                        // a K slice past the row's end adds nothing
                        acc[n][rt][r] = live ? __builtin_fmaf(yd[r], v, acc[n][rt][r]) : acc[n][rt][r];
                    }
            };
            v4i_t pl[2], ph[2];
            read_a(0u);
#pragma unroll
            for (uint32_t n = 0; n < NS; n++) {
                if (n + 1u < NS) read_a(n + 1u);
                v4i_t dl[2] = {}, dh[2] = {};
#pragma unroll
                for (uint32_t s = 0; s < 4; s++)
#pragma unroll
                    for (int rt = 0; rt < 2; rt++) {
                        dl[rt] = mfma64(a[n & 1u][s], tw[rt].lo[s], dl[rt]);
                        if (F::kHi) dh[rt] = mfma64(a[n & 1u][s], tw[rt].hi[s], dh[rt]);
                    }
                if (n > 0u) finish(n - 1u, pl, ph);
#pragma unroll
                for (int rt = 0; rt < 2; rt++) {
                    pl[rt] = dl[rt];
                    ph[rt] = dh[rt];
                }
            }
            finish(NS - 1u, pl, ph);
            arrived();
        };
        arrived();
        for (uint32_t it = 0;;) {
            step(buf0, buf1, it);
            if (++it == n_it) break;
            step(buf1, buf0, it);
            if (++it == n_it) break;
        }
        if constexpr (WK > 1) {
            // [wave][slice][tile][element][lane], two waves' partials per buffer
            static_assert(kBuf >= 2u * NS * 8u * 256u, "the partials fit the buffers");
            auto part = [&](uint32_t wv, uint32_t n, uint32_t rt, uint32_t r) {
                return (float *)(wv < 2u ? buf0 : buf1) + (((wv & 1u) * NS + n) * 8u + rt * 4u + r) * 64u + lane;
            };
#pragma unroll
            for (uint32_t n = 0; n < NS; n++)
#pragma unroll
                for (uint32_t e = 0; e < 8; e++) *part(wave, n, e >> 2, e & 3u) = acc[n][e >> 2][e & 3u];
            __syncthreads();
            const uint32_t wr = wave % WR;
#pragma unroll
            for (uint32_t n = 0; n < NS; n++)
#pragma unroll
                for (uint32_t e = 0; e < 8; e++)
                    if (mine(n, e & 3u, wk)) {
                        float v = *part(wr, n, e >> 2, e & 3u);
#pragma unroll
                        for (uint32_t k = 1; k < WK; k++) v += *part(k * WR + wr, n, e >> 2, e & 3u);
                        acc[n][e >> 2][e & 3u] = v;
                    }
            __syncthreads();
        }
    }
    // Which K slice finishes element r of slice n (both row tiles): the 4 NS
    // (slice, element) places in WK runs
    PK_DEV static bool mine(uint32_t n, uint32_t r, uint32_t wk) { return WK == 1u || (4u * n + r) * WK / (4u * NS) == wk; }
};

// Blocks in flight at once: two per CU (256 VGPRs, 160 KiB of LDS).
constexpr uint32_t kTileSlots = 512;

// The tile of the expert groups: Tile<Q, 4, 1, NS> with the order of a token
// slice's steps fixed. Its time goes to LDS reads that are waited for at once:
// at 250 registers the compiler reads a step's tokens right before their MFMAs
// (timed without those reads, a Q4_K tile of 8 slices takes 51 us instead of
// 72). Here the tokens of a step are read again, for the next slice, as soon as
// the step's MFMAs are issued, 12 MFMAs ahead of their use and into the same
// registers, with a quarter of the previous slice's fp32 step beside them.
// The lane keeps the 32-bit q8_K rows of the records it copies and forms their
// addresses, two registers each, in every iteration: half the spills. Prefill
// of 128 Q4_K / Q6_K experts, 1536 tokens top-8: 437 -> 401 us a layer; IQ2_XXS
// chunk of 100 tokens: 498 -> 485. The 16-row kernel's fp32 step, which has three
// more vector operations for formats with mins, takes the Q4_K stage of that
// layer from 210 to 220 (the layer 400 -> 411). The dense kernel keeps Tile::run: fixed in
// this order its 8-slice Q4_K tile spills 37 registers (77 -> 91 us), and its
// tiles of 2 to 4 slices take 1-2% longer.
template <uint32_t Q, uint32_t NS>
struct GroupedTile : Tile<Q, 4, 1, NS> {
    using T = Tile<Q, 4, 1, NS>;
    using F = TileFmt<Q>;

    // As Tile::run, with row_of(t): the q8_K row, of nb blocks each from xb on,
    // of token t. NC: the token slices computed (16 NC >= np).
    template <uint32_t NC, typename RowOf>
    PK_DEV void run(uint8_t *buf0, uint8_t *buf1, const uint2 *lut, const uint8_t *w0, const uint8_t *w1, uint32_t nb,
                    uint32_t np, const uint8_t *xb, RowOf row_of) {
        const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
        const uint32_t i = lane & 15u, q = lane >> 4;
        // tokens past np: the last one again
        auto row = [&](uint32_t t) { return row_of(t < np ? t : np - 1u); };
        uint32_t xrow[NS];
#pragma unroll
        for (uint32_t m = 0; m < NS; m++) xrow[m] = row(4u * (wave + 4u * m) + lane / 16u);
        const uint32_t bs_blk = T::kRec >= 128u ? wave : wave % (T::kRec / 32u), d_blk = wave % (T::kRec / 64u);
        const uint32_t bs_row = row(32u * bs_blk + lane / 2u), d_row = row(64u * d_blk + lane);
        // as Tile::run's copies
        auto dma = [&](uint8_t *buf, uint32_t it) {
            uint32_t stride = nb * 292u;
            asm volatile("" : "+s"(stride));  // the products are not hoisted out of the loop
            auto src = [&](uint32_t r, uint32_t at) {
                return (const PK_GLOBAL uint32_t *)(xb + ((it < nb ? it : nb - 1u) * 292u + at) + (uint64_t)r * stride);
            };
#pragma unroll
            for (uint32_t m = 0; m < NS; m++) {
                const uint32_t r0 = 4u * (wave + 4u * m), rec = r0 + lane / 16u;
                __builtin_amdgcn_global_load_lds(src(xrow[m], 4u + 16u * ((lane ^ rec) & 15u)),
                                                 (PK_LDS uint32_t *)(buf + r0 * 256u), 16, 0, 0);
            }
            if (F::kMin)
                __builtin_amdgcn_global_load_lds(src(bs_row, 260u + 16u * (lane & 1u)),
                                                 (PK_LDS uint32_t *)(buf + T::kBsum + 1024u * bs_blk), 16, 0, 0);
            __builtin_amdgcn_global_load_lds(src(d_row, 0u), (PK_LDS uint32_t *)(buf + T::kD + 256u * d_blk), 4, 0, 0);
        };
#pragma unroll
        for (uint32_t n = 0; n < NS; n++)
#pragma unroll
            for (int r = 0; r < 4; r++) this->acc[n][0][r] = this->acc[n][1][r] = 0.0f;
        uint32_t ao[4];  // byte offset of the lane's piece of step s, token slice 0
#pragma unroll
        for (uint32_t s = 0; s < 4; s++) ao[s] = i * 256u + 16u * (F::piece(s, q) ^ i);
        dma(buf0, 0u);
        typename F::Raw raw[2];
        auto load_w = [&](uint32_t it) {  // past the end: the last super-block again
            const uint64_t o = (uint64_t)(it < nb ? it : nb - 1u) * F::kSb;
            raw[0] = F::load(w0 + o, q);
            raw[1] = F::load(w1 + o, q);
        };
        load_w(0u);
        auto arrived = [] {
            __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0): the wave's DMA writes are in LDS
            __syncthreads();
        };
        auto step = [&](const uint8_t *buf, uint8_t *nbuf, uint32_t it) {
            TileW tw[2];
            F::decode(raw[0], q, lut, tw[0]);
            F::decode(raw[1], q, lut, tw[1]);
            __builtin_amdgcn_sched_barrier(0);
            dma(nbuf, it + 1u);
            // late where the accumulators leave few registers
            constexpr uint32_t kLoadAt = NC > 4u ? NC - 2u : 0u;
            if (kLoadAt == 0u) load_w(it + 1u);
            __builtin_amdgcn_sched_barrier(0);
            uint4 a[4];
            auto read_a = [&](uint32_t n, uint32_t s) { a[s] = *(const uint4 *)(buf + ao[s] + 4096u * n); };
            // what the fp32 step of a slice needs besides its integer sums
            struct Side {
                uint4 y;
                uint2 b;
                v4f_t ms[2];
            };
            auto read_side = [&](uint32_t n, Side &d) {
                d.y = *(const uint4 *)(buf + T::kD + (16u * n + 4u * q) * 4u);
                if constexpr (F::kMin) d.b = *(const uint2 *)(buf + T::kBsum + (16u * n + i) * 32u + 8u * q);
            };
            auto min_terms = [&](Side &d) {
                if constexpr (F::kMin) {
                    const uint2 bh = make_uint2(f16_of_i16(d.b.x), f16_of_i16(d.b.y));
                    d.ms[0] = mfma16_f16(bh, tw[0].mins);
                    d.ms[1] = mfma16_f16(bh, tw[1].mins);
                }
            };
            // the fp32 step of token 4q + r of slice n, with the products and
            // roundings of the 16-row kernel (mmq.hip): the integer sums are
            // exact in both, so a pair's value is the same whichever runs it
            auto finish = [&](uint32_t n, uint32_t r, const Side &d, const v4i_t (&dl)[2], const v4i_t (&dh)[2]) {
                const float yd = __uint_as_float(word4(d.y, r));
#pragma unroll
                for (int rt = 0; rt < 2; rt++) {
                    const int32_t sum = F::kHi ? (int32_t)((uint32_t)dh[rt][r] << F::kShift) + dl[rt][r] : dl[rt][r];
                    const float xy = (F::kNeg ? -tw[rt].xd : tw[rt].xd) * yd;
                    float &a = this->acc[n][rt][r];
                    if constexpr (F::kMin)
                        a += xy * (float)sum - tw[rt].xmin * yd * d.ms[rt][r];
                    else
                        a = __builtin_fmaf(xy, (float)sum, a);
                }
            };
            v4i_t pl[2], ph[2];
            Side ps;
#pragma unroll
            for (uint32_t s = 0; s < 4; s++) read_a(0u, s);
#pragma unroll
            for (uint32_t n = 0; n < NC; n++) {
                v4i_t dl[2] = {}, dh[2] = {};
                Side d;
                read_side(n, d);
                if (n > 0u && n == kLoadAt) load_w(it + 1u);
#pragma unroll
                for (uint32_t s = 0; s < 4; s++) {
#pragma unroll
                    for (int rt = 0; rt < 2; rt++) {
                        dl[rt] = mfma64(a[s], tw[rt].lo[s], dl[rt]);
                        if (F::kHi) dh[rt] = mfma64(a[s], tw[rt].hi[s], dh[rt]);
                    }
                    if (n + 1u < NC) read_a(n + 1u, s);
                    if (n > 0u) finish(n - 1u, s, ps, pl, ph);
                    if (s == 3u) min_terms(d);
                    __builtin_amdgcn_sched_barrier(0);
                }
#pragma unroll
                for (int rt = 0; rt < 2; rt++) {
                    pl[rt] = dl[rt];
                    ph[rt] = dh[rt];
                }
                ps = d;
            }
#pragma unroll
            for (uint32_t r = 0; r < 4; r++) finish(NC - 1u, r, ps, pl, ph);
            arrived();
            hold_raw(raw[0]);
            hold_raw(raw[1]);
        };
        arrived();
        for (uint32_t it = 0;;) {
            step(buf0, buf1, it);
            if (++it == nb) break;
            step(buf1, buf0, it);
            if (++it == nb) break;
        }
    }
};

}  // namespace pk
