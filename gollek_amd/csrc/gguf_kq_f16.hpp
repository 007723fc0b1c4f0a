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
// largest magnitude to [2^8, 2^9); bf16 elements are then exact in fp16 unless
// they are below 2^-23 of that maximum, where the error is below 2^-33 of it.
//
// Column order.  Which 8 columns of the superblock lane group g (lane >> 4)
// supplies to MFMA i is free as long as both operands agree, so it follows
// the packed bytes (kq_place): a lane's 64 codes are one contiguous run of each
// byte array, and a dword of four packed bytes gives the pairs (0, 2), (1, 3)
// with one AND each.
//
// Min term (Q4_K, Q5_K): sum_j m_j * sum(x of sub-block j) is one more MFMA:
// lane group g holds the sums of sub-blocks 2g, 2g + 1 as three fp16 digits
// each (A) against m_2g, m_2g+1 three times each (B).
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
            const _Float16 m0 = (_Float16)(unsigned short)(mnp & 0xFFu), m1 = (_Float16)(unsigned short)(mnp >> 8);
            bm = f16x8{m0, m0, m0, (_Float16)0.0f, m1, m1, m1, (_Float16)0.0f};
            if constexpr (kCentered) {
                const _Float16 c0 = (_Float16)(unsigned short)(scp & 0xFFu), c1 = (_Float16)(unsigned short)(scp >> 8);
                bs = f16x8{c0, c0, c0, (_Float16)0.0f, c1, c1, c1, (_Float16)0.0f};
            }
            d = half_bits_to_float_fast(r.hd.x & 0xFFFFu) * kq_code_scale<T>();
            // no min code set: a non-finite dmin stays out
            // (RT/GgufKQuantLayout.java:67-69)
            dm = (r.hd.z | (r.hd.w & 0xF0F0F0F0u)) != 0u ? half_bits_to_float_fast(r.hd.x >> 16) : 0.0f;
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

// max |v| < 2^(E - 126) (E: biased exponent of the largest magnitude): the
// power of two that brings it to [2^8, 2^9), and its inverse.
__device__ __forceinline__ void kq_row_scale(float mx, float &s, float &inv) {
    uint32_t e = (__float_as_uint(mx) >> 23) & 0xFFu;
    e = e < 9u ? 9u : e;
    s = __uint_as_float((262u - e) << 23);
    inv = __uint_as_float((e - 8u) << 23);
}

// t (|t| <= 2^14) as three fp16 digits (half of a lane's slots of KqOperand::bm).
__device__ __forceinline__ uint2 kq_min_digits(float t) {
    const _Float16 a = (_Float16)t;
    const float r = t - (float)a;
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
// 15) over superblocks sb_of(st) of stages [st0, st1).  `units`: the wave's
// first unit in buffer 0; buffer 1 is `flip` bytes after it.  begin() requests
// the first stage's x and ready() has it in LDS (the first raw bytes of W are
// requested between the two, so that their latencies overlap); produce(kc, st,
// buffer), called in every step (kc::value = 0 .. 7) of a stage that another one
// follows, brings the x of stage st into that buffer.
//
// A step takes 2 MT DIGITS kTerms MFMAs (one fragment of W); the next
// fragment's codes are widened while they run.  The next stage's raw bytes
// replace this stage's after their last use, in step 6 (requested a stage
// ahead into registers of their own they cost the small tiles a workgroup per
// CU: Q4_K M = 16, 14336 x 4096, 15.0 against 17.7 us).  The last stage is a copy
// of its own without either: brought in again for nobody, they cost a wait for
// x and a conversion (Q5_K M = 5, 1024 x 2048, one stage of eight slices: 8.44
// against 7.19 us; Q6_K M = 333, 4096 x 14336: 101.4 against 98.6).
template <int T, int MT, int DIGITS, bool CENTERED, class SbOf, class Begin, class Ready, class Produce>
__device__ __forceinline__ void kq_stages(f32x4 (&acc)[MT][2], const uint8_t *const (&wp)[2], const uint8_t *units,
                                          int flip, int st0, int st1, int nsb, int lane, SbOf &&sb_of,
                                          Begin &&begin, Ready &&ready, Produce &&produce) {
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
        const bool act = sb_of(st) < nsb;  // uniform
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
#pragma unroll
        for (int mt = 0; mt < MT; mt++) {
            const uint8_t *const unit = cur + mt * U::kBytes;
            const f32x4 inv = *reinterpret_cast<const f32x4 *>(unit + U::kScales + 16 * g);
            f32x4 pm[2], ps[2];
            if constexpr (Op::kMins) {
                const f16x8 am = *reinterpret_cast<const f16x8 *>(unit + U::kMins + 64 * n + 16 * g);
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
                    if constexpr (Op::kCentered) {  // d P + (d 2^-15 8 PS - dmin PM): the small part last
                        const float c = op[nt].d * (T == kQ5_K ? 0x1p-11f : 0x1p-12f);
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
    stage(st1 - 1, std::true_type{});
}

}  // namespace kqf
}  // namespace gollek
