// gguf_kq_f16.hpp -- K-quant rows as exact fp16 matrix-core operands.
//
// v_mfma_f32_16x16x32_f16 contracts x with W in fp16, whose 11-bit
// significand holds what an integer product of a K-quant superblock needs:
// Q4_K sc * q <= 63 * 15 and Q5_K sc * q <= 63 * 31 are exact in one operand;
// Q6_K's sc * (q - 32) (up to 4096) is the sum of sc * nibble (<= 1920) and
// 16 sc * (qh - 2) (256 times 16), both exact, so it takes two.  With the
// scale code inside the operand an MFMA may mix scale groups, so all 256
// columns of a superblock accumulate in the matrix cores and the fp32 factor d
// is applied once per output and superblock (the bf16 tile kernel applies one
// FMA per 32-element block, four VALU instructions per MFMA).
//
// x: each (row, superblock) is scaled by a power of two that brings its
// largest magnitude to [2^14, 2^15); bf16 elements are then exact in fp16
// unless they are below 2^-31 of that maximum, where the error is at most 2^-39
// of it.  Rows with an outlier of 2^20 times half the superblock's columns and
// more (kq_wide), and those with an infinity (the parts of a Q6_K product would cancel
// to NaN), are computed again by kq_wide_rows (Q4_K M = 512, 14336 x 4096: 229 us
// with one such row, 1030 with 512 of them, 104 with none on the same card).
//
// Column order.  Which 8 columns of the superblock lane group g (lane >> 4)
// supplies to MFMA i is free as long as both operands agree, so it follows
// the packed bytes (kq_place): a lane's 64 codes are one contiguous run of each
// byte array, and a dword of four packed bytes gives the pairs (0, 2), (1, 3)
// with one AND each.
//
// Min term (Q4_K, Q5_K): sum_j m_j * sum(x of sub-block j) is one more MFMA:
// lane group g holds the sums of sub-blocks 2g, 2g + 1 (up to 2^20, as 2^-6 of
// that) as three fp16 digits each (A), the second and third times 2^12, against
// m_2g, m_2g+1 once and twice times 2^-12 (B).
#pragma once

#include <type_traits>
#include <utility>

#include "gguf_blocks.hpp"
#include "gguf_kernels.hpp"

namespace gollek {
namespace kqf {

typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t v4u __attribute__((ext_vector_type(4)));

// Unaligned 16- and 8-byte loads (superblocks start on even bytes).
struct __attribute__((packed, aligned(2))) Bytes16 {
    uint32_t v[4];
};
struct __attribute__((packed, aligned(2))) Bytes8 {
    uint32_t v[2];
};
__device__ __forceinline__ v4u ld16(const uint8_t *p) {
    const Bytes16 b = *reinterpret_cast<const Bytes16 *>(p);
    return v4u{b.v[0], b.v[1], b.v[2], b.v[3]};
}

__device__ __forceinline__ f32x4 mfma_f16(f16x8 a, f16x8 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
}

template <int T>
constexpr int kq_block_bytes() {
    return T == kQ6_K ? 210 : T == kQ5_K ? kQ5KBlockBytes : kQKBlockBytes;
}
// Power of two the operand products carry (undone in d).
template <int T>
constexpr float kq_code_scale() {
    return T == kQ6_K ? 0x1p16f : 0x1p15f;
}

// MFMA of step k (0 .. 7) of a superblock: the order uses up the first half of
// the code bytes first.  Q4_K / Q5_K: 0, 4, 1, 5, ...; Q6_K: quarters 0, 2, 1,
// 3 of a half, two each.
template <int T>
__device__ __forceinline__ constexpr int kq_order(int k) {
    return T == kQ6_K ? (k < 2 ? k : k < 4 ? k + 2 : k < 6 ? k - 2 : k) : (k & 1) * 4 + (k >> 1);
}
template <int T>
__device__ __forceinline__ constexpr int kq_step(int i) {  // its inverse
    return T == kQ6_K ? (i < 2 ? i : i < 4 ? i + 2 : i < 6 ? i - 2 : i) : 2 * (i & 3) + (i >> 2);
}

// Lane group and steps of the 16 superblock columns from 16 c: the first 8
// belong to step k0 and the rest to step k1 of the same half (k0 / 4 == k1 /
// 4).  A lane's 8 slots hold columns + 0, 2, 1, 3, 4, 6, 5, 7.
template <int T>
__device__ __forceinline__ void kq_place(int c, int &g, int &k0, int &k1) {
    const int i = T == kQ6_K ? 2 * ((c >> 1) & 3) : 2 * (c & 3);
    g = T == kQ6_K ? 2 * (c >> 3) + (c & 1) : c >> 2;
    k0 = kq_step<T>(i);
    k1 = kq_step<T>(i + 1);
}

// A lane's raw bytes of one superblock (row lane & 15 of a 16-row tile, lane
// group g), loaded in parts so that the next superblock's bytes can replace
// them as they are used up.  Q4_K / Q5_K: the header, the 32 quant bytes of
// chunk g (and the 32 qh bytes); Q6_K: 16 bytes each of the half's two ql runs
// and of qh, the half's 8 scales, d.
template <int T>
struct KqRaw {
    v4u hd, q0, q1, h0, h1;
    __device__ __forceinline__ void load_head(const uint8_t *p, int) { hd = ld16(p); }
    // Q4_K / Q5_K: the quants (and qh bytes) of MFMAs 4 + (2 half, + 1) and (2 half, + 1)
    template <int HALF>
    __device__ __forceinline__ void load_codes(const uint8_t *p, int g) {
        const uint8_t *q = p + (T == kQ5_K ? 48 : 16) + 32 * g + 16 * HALF;
        if constexpr (T == kQ5_K) (HALF ? h1 : h0) = ld16(p + 16 + 16 * HALF);
        (HALF ? q1 : q0) = ld16(q);
    }
};
template <>
struct KqRaw<kQ6_K> {
    v4u q0, q1, h0;
    uint32_t s0, s1, d;
    __device__ __forceinline__ void load_head(const uint8_t *p, int g) {
        const Bytes8 s = *reinterpret_cast<const Bytes8 *>(p + 192 + 8 * (g >> 1));
        s0 = s.v[0];
        s1 = s.v[1];
        d = *reinterpret_cast<const uint16_t *>(p + 208);
    }
    // half 0: the run of quarters 0, 2 and qh; half 1: the run of quarters 1, 3
    template <int HALF>
    __device__ __forceinline__ void load_codes(const uint8_t *p, int g) {
        const int h = g >> 1, l0 = 16 * (g & 1);
        (HALF ? q1 : q0) = ld16(p + 64 * h + 32 * HALF + l0);
        if constexpr (HALF == 1) h0 = ld16(p + 128 + 32 * h + l0);
    }
};

__device__ __forceinline__ f16x2 as_h2(uint32_t v) { return __builtin_bit_cast(f16x2, v); }
__device__ __forceinline__ uint32_t as_u(f16x2 v) { return __builtin_bit_cast(uint32_t, v); }
__device__ __forceinline__ f16x8 as_h8(const uint32_t (&v)[4]) {
    return __builtin_bit_cast(f16x8, v4u{v[0], v[1], v[2], v[3]});
}
__device__ __forceinline__ f16x2 splat(_Float16 v) { return f16x2{v, v}; }

// Two codes (bytes 0 and 1 of w) against kq_min_digits: v, v 2^-12, v 2^-12
// each (an integer v is the fp16 subnormal v 2^-24).
__device__ __forceinline__ f16x8 kq_digit_codes(uint32_t w) {
    const f16x2 b = as_h2((w & 0xFFu) | (w >> 8) << 16) * splat((_Float16)0x1p12f), a = b * splat((_Float16)0x1p12f);
    const _Float16 z = (_Float16)0.0f;
    return f16x8{a[0], b[0], b[0], z, a[1], b[1], b[1], z};
}

// One 16-row tile's operand of a superblock.  head() decodes the row's scale
// codes, the min operand and the fp32 factors; frag() the codes of one MFMA
// (kTerms operands) from the raw bytes.
//
// Codes enter as fp16 subnormals (the integer q has the value q 2^-24, a high
// nibble in place 16 q 2^-24), so widening two of them is one AND and the
// multiplication by the scale code is also the conversion:
// q 2^-24 * (sc 2^9) = sc q 2^-15, exact (11 bits above 2^-24).
//
// CENTERED (Q4_K, Q5_K): the operand is sc (q - 8) (Q5_K: q - 16; still exact)
// and d * 8 (16) * sum_j sc_j * sum(x of sub-block j), one more MFMA like the
// min term, is added back.  The codes' mean makes up most of an uncentered
// sum, which then cancels against the min term, so its roundings count about
// three times as much.
template <int T, bool CENTERED>
struct KqOperand {
    static constexpr int kTerms = T == kQ6_K ? 2 : 1;
    static constexpr bool kMins = T != kQ6_K;
    static constexpr bool kCentered = CENTERED && kMins;
    f16x2 s[T == kQ6_K ? 4 : 2];  // scale codes as operand factors
    f16x8 bm, bs;
    float d, dm;
    __device__ __forceinline__ void head(const KqRaw<T> &r, int g) {
        if constexpr (T == kQ6_K) {
#pragma unroll
            for (int j = 0; j < 4; j++) {  // scale 2 j + (g & 1) of the half's eight
                const uint32_t w = (j & 2) ? r.s1 : r.s0;
                const int sc = (int)(int8_t)(w >> (16 * (j & 1) + 8 * (g & 1)));
                s[j] = splat((_Float16)(short)(sc * 256));
            }
            d = half_bits_to_float_fast(r.d) * kq_code_scale<T>();
            dm = 0.0f;
        } else {
            uint32_t scp, mnp;
            q4k_pair_codes(r.hd.y, r.hd.z, r.hd.w, g, &scp, &mnp);
            s[0] = splat((_Float16)(unsigned short)((scp & 0xFFu) << 9));
            s[1] = splat((_Float16)(unsigned short)((scp >> 8) << 5));
            bm = kq_digit_codes(mnp);
            if constexpr (kCentered) bs = kq_digit_codes(scp);
            d = half_bits_to_float_fast(r.hd.x & 0xFFFFu) * kq_code_scale<T>();
            // no min code set: a non-finite dmin stays out
            // (RT/GgufKQuantLayout.java:67-69)
            dm = (r.hd.z | (r.hd.w & 0xF0F0F0F0u)) != 0u ? half_bits_to_float_fast(r.hd.x >> 16) * 0x1p6f : 0.0f;
        }
    }
    __device__ __forceinline__ void frag(const KqRaw<T> &r, int g, int i, f16x8 (&b)[kTerms]) const {
        uint32_t lo[4], hi[4];
        if constexpr (T == kQ6_K) {
            const int j = i >> 1, hf = i & 1;
            const f16x2 sn = (j & 2) ? s[j] * splat((_Float16)0x1p-4f) : s[j];
            const f16x2 c = s[j] * splat((_Float16)-0x1p-19f);  // -32 sc 2^-16
#pragma unroll
            for (int t = 0; t < 2; t++) {
                const int k = 2 * hf + t;
                const uint32_t q = (j & 1) ? r.q1[k] : r.q0[k], h = r.h0[k];
                const uint32_t mask = (j & 2) ? 0x00F000F0u : 0x000F000Fu;
                lo[2 * t] = as_u(as_h2(q & mask) * sn);
                lo[2 * t + 1] = as_u(as_h2((q >> 8) & mask) * sn);
                const uint32_t he = j == 0 ? h << 4 : j == 1 ? h << 2 : j == 2 ? h : h >> 2;
                const uint32_t ho = j == 0 ? h >> 4 : j == 1 ? h >> 6 : j == 2 ? h >> 8 : h >> 10;
                hi[2 * t] = as_u(__builtin_elementwise_fma(as_h2(he & 0x00300030u), s[j], c));
                hi[2 * t + 1] = as_u(__builtin_elementwise_fma(as_h2(ho & 0x00300030u), s[j], c));
            }
            b[kTerms - 1] = as_h8(hi);
        } else {
            const bool up = i >= 4;  // sub-block 2g + 1: the high nibbles
            const uint32_t mask = up ? 0x00F000F0u : 0x000F000Fu;
#pragma unroll
            for (int t = 0; t < 2; t++) {
                const int k = 2 * (i & 3) + t;
                const uint32_t q = k < 4 ? r.q0[k & 3] : r.q1[k & 3];
                uint32_t u0 = q & mask, u1 = (q >> 8) & mask;
                if constexpr (T == kQ5_K) {
                    const uint32_t h = (k < 4 ? r.h0[k & 3] : r.h1[k & 3]) >> (2 * g);
                    u0 |= up ? (h << 7) & 0x01000100u : (h << 4) & 0x00100010u;
                    u1 |= up ? (h >> 1) & 0x01000100u : (h >> 4) & 0x00100010u;
                }
                if constexpr (kCentered) {  // s = sc 2^9 (low) or sc 2^5: -8 sc 2^-15, Q5_K -16 sc 2^-15
                    const f16x2 c = s[up] * splat((_Float16)((up ? -0x1p-17f : -0x1p-21f) * (T == kQ5_K ? 2.0f : 1.0f)));
                    lo[2 * t] = as_u(__builtin_elementwise_fma(as_h2(u0), s[up], c));
                    lo[2 * t + 1] = as_u(__builtin_elementwise_fma(as_h2(u1), s[up], c));
                } else {
                    lo[2 * t] = as_u(as_h2(u0) * s[up]);
                    lo[2 * t + 1] = as_u(as_h2(u1) * s[up]);
                }
            }
        }
        b[0] = as_h8(lo);
    }
};

// The x operand of 16 rows and one superblock (a unit), as it stands in LDS:
// per half (steps 0 .. 3, 4 .. 7) and digit 256 bytes a row, its pieces (16
// bytes: one lane's slots of a step), piece 4 (k & 3) + g at 16-byte position
// piece ^ row (so the 16 rows a fragment read touches hit distinct banks);
// then the rows' min pieces and their inverse scales.
template <int DIGITS>
struct KqUnit {
    static constexpr int kDigit = 16 * 256, kHalf = kDigit * DIGITS;
    static constexpr int kMins = 2 * kHalf;         // 4 pieces a row, by lane group
    static constexpr int kScales = kMins + 16 * 64;
    static constexpr int kBytes = kScales + 64;
    __device__ static __forceinline__ int piece(int k, int g, int row) {
        return kHalf * (k >> 2) + 256 * row + 16 * ((4 * (k & 3) + g) ^ row);
    }
};

template <int CTRL>
__device__ __forceinline__ float kq_dpp(float v) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xF, 0xF, true));
}
// Maximum over the 16 lanes of a DPP row.
__device__ __forceinline__ float row_max16(float v) {
    v = fmaxf(v, kq_dpp<0xB1>(v));   // quad_perm [1,0,3,2]
    v = fmaxf(v, kq_dpp<0x4E>(v));   // quad_perm [2,3,0,1]
    v = fmaxf(v, kq_dpp<0x124>(v));  // row_ror:4
    return fmaxf(v, kq_dpp<0x128>(v));  // row_ror:8
}

// For a row's superblock whose largest magnitude is mx: the power of two that
// brings it to [2^14, 2^15), and its inverse (magnitudes below 2^-106 are scaled
// as that one, so that kq_wide's bound is a normal number).
__device__ __forceinline__ void kq_row_scale(float mx, float &s, float &inv) {
    uint32_t e = __float_as_uint(mx) & 0x7F800000u;
    e = e < (21u << 23) ? 21u << 23 : e;
    s = __uint_as_float((268u << 23) - e);
    inv = __uint_as_float(e - (14u << 23));
}

// Whether a row's superblock of maximum `mx` is one for kq_wide_rows: an
// infinity, or kWideRuns of its 16 runs of 16 columns each of a maximum
// (`lane_mx`) that is not 0 and below 2^-6 when scaled, where fp16's rounding is
// 2^-19 of it (an outlier of 2^20 times the rest, its weights 0: 1.5e-7 of error in
// the result, fp32 sums of K = 2048 1 to 6e-7).  Fewer such runs are no outlier's
// superblock but the tails of a gated activation beside values that outweigh
// them by 2^20.  The lanes that find one (a ballot each: of the two together it
// takes a select and a second comparison); an infinity counts in all 16.
constexpr int kWideRuns = 8;
__device__ __forceinline__ uint64_t kq_wide(float lane_mx, float mx, float inv) {
    return __builtin_amdgcn_ballot_w64(__float_as_uint(lane_mx) - 1u < __float_as_uint(inv) - (6u << 23)) |
           __builtin_amdgcn_ballot_w64(mx == __builtin_inff());
}

// t (|t| <= 2^14) as three fp16 digits, the second and third times 2^12 (half of
// a lane's slots of KqOperand::bm).
__device__ __forceinline__ uint2 kq_min_digits(float t) {
    const _Float16 a = (_Float16)t;
    const float r = (t - (float)a) * 0x1p12f;
    const _Float16 b = (_Float16)r;
    const _Float16 c = (_Float16)(r - (float)b);
    return uint2{as_u(f16x2{a, b}), as_u(f16x2{c, (_Float16)0.0f})};
}

template <class F, int... I>
__device__ __forceinline__ void static_for_impl(F &&f, std::integer_sequence<int, I...>) {
    (f(std::integral_constant<int, I>{}), ...);
}
template <int N, class F>
__device__ __forceinline__ void static_for(F &&f) {
    static_for_impl(f, std::make_integer_sequence<int, N>{});
}

// The stage loop: acc[mt][nt] += the contraction of the workgroup's MT row
// tiles with this wave's two 16-row tiles of W (rows wp[0], wp[1] at lane &
// 15) over superblocks sb_of(st) of stages [st0, st1) (WHOLE: none is past the
// last; otherwise selects, 64 of the 870 VALU instructions of a 128-row stage,
// keep those out).  `units`: the wave's first unit in buffer 0; buffer 1 is `flip`
// bytes after it.  begin() requests the first stage's x and ready() has it in LDS
// (the first raw bytes of W are requested between the two, so that their
// latencies overlap); produce(kc, st, buffer), called in every step (kc::value =
// 0 .. 7) of a stage that another one follows, brings the x of stage st into that
// buffer; done() runs before the last stage, whose barrier publishes what it
// writes to LDS.
//
// A step takes 2 MT DIGITS kTerms MFMAs (one fragment of W); the next
// fragment's codes are widened while they run.  The next stage's raw bytes
// replace this stage's after their last use, in step 6 (requested a stage
// ahead into registers of their own they cost the small tiles a workgroup per
// CU: Q4_K M = 16, 14336 x 4096, 15.0 against 17.7 us).  The last stage is a copy
// of its own without either: brought in again for nobody, they cost a wait for
// x and a conversion (Q5_K M = 5, 1024 x 2048, one stage of eight slices: 8.44
// against 7.19 us; Q6_K M = 333, 4096 x 14336: 101.4 against 98.6).
template <int T, int MT, int DIGITS, bool CENTERED, bool WHOLE, class SbOf, class Begin, class Ready, class Produce, class Done>
__device__ __forceinline__ void kq_stages(f32x4 (&acc)[MT][2], const uint8_t *const (&wp)[2], const uint8_t *units,
                                          int flip, int st0, int st1, int nsb, int lane, SbOf &&sb_of,
                                          Begin &&begin, Ready &&ready, Produce &&produce, Done &&done) {
    using Op = KqOperand<T, CENTERED>;
    using U = KqUnit<DIGITS>;
    constexpr int NT = Op::kTerms;
    constexpr int MH = MT > 4 ? MT / 2 : MT;  // row tiles whose fragments are held at a time
    constexpr int HN = MT / MH;
    const int g = lane >> 4, n = lane & 15;
    const f32x4 zero = {0.0f, 0.0f, 0.0f, 0.0f};
    int ap[4];  // the lane's piece of step k & 3
#pragma unroll
    for (int k = 0; k < 4; k++) ap[k] = U::piece(k, g, n);
    KqRaw<T> raw[2];
    auto load_w = [&](int st) {
        const int sb = sb_of(st);
#pragma unroll
        for (int nt = 0; nt < 2; nt++) {
            const uint8_t *const p = wp[nt] + (int64_t)(sb < nsb ? sb : nsb - 1) * kq_block_bytes<T>();
            raw[nt].load_head(p, g);
            raw[nt].template load_codes<0>(p, g);
            raw[nt].template load_codes<1>(p, g);
        }
    };
    begin();
    load_w(st0);
    ready();
    auto stage = [&](int st, auto last) {
        const uint8_t *const cur = units + ((st - st0) & 1) * flip;
        f32x4 p[MT][2];
        Op op[2];
        f16x8 b[2][2][NT];
#pragma unroll
        for (int nt = 0; nt < 2; nt++) {
            op[nt].head(raw[nt], g);
            op[nt].frag(raw[nt], g, kq_order<T>(0), b[0][nt]);
        }
        const bool act = WHOLE || sb_of(st) < nsb;  // uniform
        static_for<8>([&](auto kc) {
            constexpr int k = kc.value;
            static_for<DIGITS * HN>([&](auto hc) {
                constexpr int dg = hc.value / HN, h = hc.value % HN;
                f16x8 a[MH];
#pragma unroll
                for (int mt = 0; mt < MH; mt++)
                    a[mt] = *reinterpret_cast<const f16x8 *>(cur + (h * MH + mt) * U::kBytes + U::kDigit * dg +
                                                             U::kHalf * (k >> 2) + ap[k & 3]);
#pragma unroll
                for (int q = 0; q < NT; q++)
#pragma unroll
                    for (int mt = 0; mt < MH; mt++)
#pragma unroll
                        for (int nt = 0; nt < 2; nt++) {
                            f32x4 &c = p[h * MH + mt][nt];
                            c = mfma_f16(a[mt], b[k & 1][nt][q], k == 0 && dg == 0 && q == 0 ? zero : c);
                        }
                if constexpr (k < 7) {
                    constexpr int R = DIGITS * HN;
                    if constexpr (hc.value == 0) op[0].frag(raw[0], g, kq_order<T>(k + 1), b[(k + 1) & 1][0]);
                    if constexpr (hc.value == R - 1) op[1].frag(raw[1], g, kq_order<T>(k + 1), b[(k + 1) & 1][1]);
                }
                if constexpr (hc.value == DIGITS * HN - 1 && !last.value) {
                    if constexpr (k == 6) load_w(st + 1);
                    produce(kc, st + 1, (st + 1 - st0) & 1);
                }
                // fragment reads, then the widening and conversion between the MFMAs
                __builtin_amdgcn_sched_group_barrier(0x100, MH, 0);
#pragma unroll
                for (int z = 0; z < 2 * MH * NT; z++) {
                    __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);
                    __builtin_amdgcn_sched_group_barrier(0x2, 4, 0);
                }
                __builtin_amdgcn_sched_barrier(0);
            });
        });
        int eg = g, en = n;
        if constexpr (T == kQ4_K && MT == 8) {  // no registers for offsets that are kept through the stage
            int l = lane;
            asm volatile("" : "+v"(l));
            eg = l >> 4;
            en = l & 15;
        }
#pragma unroll
        for (int mt = 0; mt < MT; mt++) {
            const uint8_t *const unit = cur + mt * U::kBytes;
            const f32x4 inv = *reinterpret_cast<const f32x4 *>(unit + U::kScales + 16 * eg);
            f32x4 pm[2], ps[2];
            if constexpr (Op::kMins) {
                const f16x8 am = *reinterpret_cast<const f16x8 *>(unit + U::kMins + 64 * en + 16 * eg);
#pragma unroll
                for (int nt = 0; nt < 2; nt++) {
                    pm[nt] = mfma_f16(am, op[nt].bm, zero);
                    if constexpr (Op::kCentered) ps[nt] = mfma_f16(am, op[nt].bs, zero);
                }
            }
#pragma unroll
            for (int nt = 0; nt < 2; nt++)
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    float v = p[mt][nt][r];
                    if constexpr (Op::kCentered) {  // d P + (d 2^-15 8 PS 2^6 - dmin PM 2^6): the small part last
                        const float c = op[nt].d * (T == kQ5_K ? 0x1p-5f : 0x1p-6f);
                        v = fmaf(op[nt].d, v, fmaf(c, ps[nt][r], -op[nt].dm * pm[nt][r]));
                    } else {
                        v *= op[nt].d;
                        if constexpr (Op::kMins) v = fmaf(-op[nt].dm, pm[nt][r], v);
                    }
                    const float c = acc[mt][nt][r];
                    acc[mt][nt][r] = act ? fmaf(inv[r], v, c) : c;
                }
        }
        __syncthreads();
    };
    for (int st = st0; st < st1 - 1; st++) stage(st, std::false_type{});
    done();
    stage(st1 - 1, std::true_type{});
}

// acc of the rows whose bit is set in `wide` (16 MT bits, the same in all waves),
// over the stages that kq_stages contracted, from dequantized weights on the fp32
// matrix cores, whole row tiles at a time.  Lane group g takes 64 columns of a
// superblock, of x and W alike: load_x(row, superblock, c, v) columns 16 c .. + 15
// of a row of the tile, and W's as its raw bytes stand.  Seldom called, so its
// loops are left rolled: it has to fit the registers that the stages leave.
template <int T, int MT, class SbOf, class LoadX>
__device__ __forceinline__ void kq_wide_rows(const uint32_t *wide, f32x4 (&acc)[MT][2], const uint8_t *const (&wp)[2],
                                             int st0, int st1, int nsb, int lane, SbOf &&sb_of, LoadX &&load_x) {
    const int g = lane >> 4, n = lane & 15;
#pragma unroll 1
    for (int mt = 0; mt < MT; mt++) {
        const uint32_t bits = (uint32_t)__builtin_amdgcn_readfirstlane((int)((wide[mt >> 1] >> (16 * (mt & 1))) & 0xFFFFu));
        if (bits == 0u) continue;
        f32x4 y[2] = {f32x4{0.0f, 0.0f, 0.0f, 0.0f}, f32x4{0.0f, 0.0f, 0.0f, 0.0f}};
#pragma unroll 1
        for (int st = st0; st < st1; st++) {
            const int sb = sb_of(st);
            if (sb >= nsb) break;
#pragma unroll 1
            for (int t = 0; t < 4; t++) {  // 16 columns: nibble t >> 1 of byte run t & 1
                float v[16];
                load_x(16 * mt + n, sb, T == kQ6_K ? 8 * (g >> 1) + 2 * t + (g & 1) : 4 * g + t, v);
#pragma unroll
                for (int nt = 0; nt < 2; nt++) {
                    __builtin_amdgcn_sched_barrier(0);
                    f32x4 part = {0.0f, 0.0f, 0.0f, 0.0f};  // (one running sum has four times the error)
                    const uint8_t *const p = wp[nt] + (int64_t)sb * kq_block_bytes<T>();
                    KqRaw<T> r;
                    r.load_head(p, g);
                    r.template load_codes<0>(p, g);
                    r.template load_codes<1>(p, g);
                    float s, m = 0.0f;  // the 16 columns' d sc and dmin m
                    if constexpr (T == kQ6_K) {
                        const uint32_t w = (t & 2) ? r.s1 : r.s0;
                        s = half_bits_to_float_fast(r.d) * (float)(int8_t)(w >> (16 * (t & 1) + 8 * (g & 1)));
                    } else {
                        uint32_t scp, mnp;
                        q4k_pair_codes(r.hd.y, r.hd.z, r.hd.w, g, &scp, &mnp);
                        const uint32_t mc = (mnp >> (8 * (t >> 1))) & 0xFFu;
                        s = half_bits_to_float_fast(r.hd.x & 0xFFFFu) * (float)((scp >> (8 * (t >> 1))) & 0xFFu);
                        m = mc ? half_bits_to_float_fast(r.hd.x >> 16) * (float)mc : 0.0f;
                    }
#pragma unroll
                    for (int i = 0; i < 16; i++) {
                        const int k = i >> 2, at = 8 * (i & 3);
                        int q = (int)((((t & 1) ? r.q1[k] : r.q0[k]) >> (at + 4 * (t >> 1))) & 15u);
                        if constexpr (T == kQ5_K)
                            q |= (int)((((t & 1) ? r.h1[k] : r.h0[k]) >> (at + 2 * g + (t >> 1))) & 1u) << 4;
                        if constexpr (T == kQ6_K) q = (q | (int)((r.h0[k] >> (at + 2 * t)) & 3u) << 4) - 32;
                        part = __builtin_amdgcn_mfma_f32_16x16x4f32(v[i], s * (float)q - m, part, 0, 0, 0);
                    }
                    y[nt] += part;
                }
            }
        }
#pragma unroll
        for (int j = 0; j < MT; j++)
#pragma unroll
            for (int r = 0; r < 4; r++)
                if (j == mt && ((bits >> (4 * g + r)) & 1u) != 0u) {
                    acc[j][0][r] = y[0][r];
                    acc[j][1][r] = y[1][r];
                }
    }
}

}  // namespace kqf
}  // namespace gollek
