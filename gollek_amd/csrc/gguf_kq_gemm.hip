// gguf_kq_gemm.hip -- GEMM Y = X . W^T for Q4_K, Q5_K and Q6_K weights on the
// fp16 matrix cores (gguf_kq_f16.hpp), X bf16 (row-major M x K), fp32
// accumulate; semantics as gguf_gemm_tile.hip (Q4_K: RT/GgufQ4RawDot.java:331-674).
//
// What bounds it: above M ~ 256 MFMA and VALU issue, whose phases in a
// workgroup's waves hardly overlap (Q4_K M = 512: 0.29 and 0.42 of the time).  A
// wave's 32 columns of a superblock take 18 MFMAs per row tile (16 cycles each)
// and, at 128 rows, per MFMA 5.6 VALU instructions: 1.6 to widen the codes, 2.3 to
// scale and convert x, 0.9 to apply d, min and the row scale; timing copies of an
// earlier form (345 us at Q4_K M = 2048, 14336 x 4096) ran in 270 without the x
// conversion, in 273 without the MFMAs.  Below that the latency of a stage (the
// next superblock's bytes are requested late in it), so small M takes small
// tiles with the superblocks spread over the waves.
// Against the bf16 kernel with one FMA per 32 columns and output that this
// replaces: Q4_K M = 2048 463 -> 338 us (711 TFLOP/s), M = 512 134 -> 85; Q6_K M =
// 333, 4096 x 14336 181 -> 99 us (its scale groups of 16 took three half-empty
// MFMAs); Q4_K M = 16 19.3 -> 15.1 us a layer of four (the first raw bytes of W
// requested only once the first x stood in LDS: 1 us more).
#include "gguf_dot4.hpp"
#include "gguf_gemm_plan.hpp"
#include "gguf_kq_f16.hpp"

namespace gollek {

using namespace kqf;

namespace {

// The x operand of one unit, four rows at a time: lane l takes columns 16 (l &
// 15) .. + 15 of row 4 j + (l >> 4) (so the loads are whole lines of X), the
// 16 lanes of a row agree on its scale, and each writes its two fragment
// pieces and its sub-block's digits.
template <int T>
struct XRows {
    v4u x[2];
    __device__ __forceinline__ void load(const uint16_t *p) {
        x[0] = *reinterpret_cast<const v4u *>(p);
        x[1] = *reinterpret_cast<const v4u *>(p + 8);
    }
    __device__ __forceinline__ void load(__amdgpu_buffer_rsrc_t rs, uint32_t off) {
        x[0] = __builtin_amdgcn_raw_buffer_load_b128(rs, off, 0, 0);
        x[1] = __builtin_amdgcn_raw_buffer_load_b128(rs, off, 16, 0);
    }
    // p0, p1: the lane's two pieces, mins: its sub-block's half of a min piece;
    // returns the lanes that find their row a wide one, if enough of them do
    __device__ __forceinline__ uint64_t store(uint8_t *p0, uint8_t *p1, uint8_t *mins, float *scale, int lane) const {
        float v[16], mx = 0.0f;
#pragma unroll
        for (int i = 0; i < 16; i++) {
            const uint32_t w = x[i >> 3][(i >> 1) & 3];
            v[i] = __uint_as_float((i & 1) ? w & 0xFFFF0000u : w << 16);
        }
#pragma unroll
        for (int i = 0; i < 16; i += 2) mx = fmaxf(fmaxf(mx, fabsf(v[i])), fabsf(v[i + 1]));
        const float lane_mx = mx;
        mx = row_max16(mx);
        float s, inv, t = 0.0f;
        kq_row_scale(mx, s, inv);
#pragma unroll
        for (int h = 0; h < 2; h++) {
            uint32_t f[4];
#pragma unroll
            for (int j = 0; j < 4; j++) {
                const int e = 8 * h + 4 * (j >> 1) + (j & 1);
                const f16x2 c = {(_Float16)(v[e] * s), (_Float16)(v[e + 2] * s)};
                f[j] = as_u(c);
                if constexpr (KqOperand<T, false>::kMins) t = __builtin_amdgcn_fdot2(c, splat((_Float16)0x1p-6f), t, false);
            }
            *reinterpret_cast<f16x8 *>(h ? p1 : p0) = as_h8(f);
        }
        if constexpr (KqOperand<T, false>::kMins) {
            t += kq_dpp<0xB1>(t);  // the sub-block's other 16 columns
            *reinterpret_cast<uint2 *>(mins) = kq_min_digits(t);  // both lanes write the same 8 bytes
        }
        if ((lane & 15) == 0) *scale = inv;
        const uint64_t found = kq_wide(lane_mx, mx, inv);
        return __builtin_popcountll(found) >= kWideRuns ? found : 0u;  // (of the four rows together)
    }
};

}  // namespace

// A workgroup owns 16 MT rows of X and 32 NW rows of W: NW KW waves as NW
// column groups of 32 and KW slices of the stage's superblocks.  Each wave
// converts its rows' share of the next stage's x between its MFMAs.
template <int T, int MT, int NW, int KW>
__global__ __launch_bounds__(64 * NW *KW, MT == 1 && NW == 2 ? 4 : 1) void gemm_kq_kernel(const uint8_t *__restrict__ W, int64_t row_bytes,
                                                              const uint16_t *__restrict__ X, float *__restrict__ Y,
                                                              int M, int N, int K, int S, float *__restrict__ part) {
    constexpr int kWaves = NW * KW, UN = MT * KW;
    constexpr int kTileM = 16 * MT, kTileN = 32 * NW;
    using U = KqUnit<1>;
    __shared__ __attribute__((aligned(16))) uint8_t lds[2][UN * U::kBytes];
    __shared__ uint32_t wide[(kTileM + 31) / 32];  // the tile's rows for kq_wide_rows

    if (threadIdx.x < (kTileM + 31) / 32) wide[threadIdx.x] = 0u;
    const int lane = (int)threadIdx.x & 63, n = lane & 15, g = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int nw = wave % NW, kw = wave / NW;

    const int tm = (M + kTileM - 1) / kTileM, tn = (N + kTileN - 1) / kTileN;
    const int G8 = (int)gridDim.x;
    const int v = (G8 % 8 == 0) ? (int)(blockIdx.x % 8) * (G8 / 8) + (int)(blockIdx.x / 8) : (int)blockIdx.x;
    const int split = v / (tm * tn);
    const int t = v - split * tm * tn;
    const int grp = t / (4 * tn);
    const int first_m = 4 * grp;
    const int gm = tm - first_m < 4 ? tm - first_m : 4;
    const int local = t - grp * 4 * tn;
    const int m0 = (first_m + local % gm) * kTileM, n0 = (local / gm) * kTileN;

    const int nsb = K / kQK, nst = (nsb + KW - 1) / KW;
    const int st0 = split * nst / S, st1 = (split + 1) * nst / S;

    const int col0 = n0 + 32 * nw;
    const uint8_t *wp[2];
#pragma unroll
    for (int nt = 0; nt < 2; nt++) {
        const int r = col0 + 16 * nt + n;
        wp[nt] = W + (int64_t)(r < N ? r : N - 1) * row_bytes;
    }
    f32x4 acc[MT][2];
#pragma unroll
    for (int mt = 0; mt < MT; mt++)
#pragma unroll
        for (int nt = 0; nt < 2; nt++) acc[mt][nt] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};

    auto sb_of = [&](int st) { return st * KW + kw; };

    // This wave's quads of rows: q = wave + kWaves j of the stage's 4 UN.
    constexpr int kPer = 4 * UN / kWaves;
    static_assert(4 * UN % kWaves == 0 && kPer <= 4, "whole quads per wave");
    int xg, xk0, xk1;
    kq_place<T>(n, xg, xk0, xk1);
    XRows<T> xr[2];
    uint64_t found[kPer] = {};
    // Q4_K's 128-row tile has no registers for four row pointers (they and the
    // epilogue's LDS offsets, spilled, were waited for with W's bytes behind them: M =
    // 512, 14336 x 4096, 89.2 against 84.7 us): it reads its rows of X through a
    // descriptor, one lane offset and a wave's, kept out of the loop's carried
    // registers; rows past M read as zeros.  Q5_K's measured 1 % slower so, Q6_K's
    // 1.2 times (it spills inside the loop).
    constexpr bool kDescriptor = T == kQ4_K && MT == 8;
    const __amdgpu_buffer_rsrc_t xs =
        wave_buffer(reinterpret_cast<const uint8_t *>(X + (int64_t)m0 * K),
                    kDescriptor ? 2u * (uint32_t)(M - m0 < kTileM ? M - m0 : kTileM) * (uint32_t)K : 0u);
    const uint32_t xo = 2u * ((uint32_t)g * (uint32_t)K + 16u * (uint32_t)n);
    auto load_x = [&](XRows<T> &to, int j, int st) {
        const int q = wave + kWaves * j, u = q >> 2, sb = st * KW + u / MT;
        if constexpr (kDescriptor) {
            uint32_t at = 2u * ((uint32_t)(16 * (u % MT) + 4 * (q & 3)) * (uint32_t)K +
                                (uint32_t)((sb < nsb ? sb : nsb - 1) * kQK));
            asm volatile("" : "+s"(at));
            to.load(xs, xo + at);
        } else {
            const int r = m0 + 16 * (u % MT) + 4 * (q & 3) + g;
            // (rows past M repeat row M - 1; their results are not stored)
            to.load(X + (int64_t)(r < M ? r : M - 1) * K + (int64_t)(sb < nsb ? sb : nsb - 1) * kQK + 16 * n);
        }
    };
    auto store_x = [&](const XRows<T> &from, int j, int b) {
        const int q = wave + kWaves * j, u = q >> 2, lr = 4 * (q & 3) + g;
        uint8_t *const unit = &lds[b][u * U::kBytes];
        found[j] |= from.store(unit + U::piece(xk0, xg, lr), unit + U::piece(xk1, xg, lr),
                               unit + U::kMins + 64 * lr + 16 * (n >> 2) + 8 * ((n >> 1) & 1),
                               reinterpret_cast<float *>(unit + U::kScales) + lr, lane);
    };
    XRows<T> first[kPer];
    kq_stages<T, MT, 1, false, KW == 1>(
        acc, wp, &lds[0][kw * MT * U::kBytes], UN * U::kBytes, st0, st1, nsb, lane, sb_of,
        [&] {
#pragma unroll
            for (int j = 0; j < kPer; j++) load_x(first[j], j, st0);
        },
        [&] {
#pragma unroll
            for (int j = 0; j < kPer; j++) store_x(first[j], j, 0);
            __syncthreads();
        },
        [&](auto kc, int st, int b) {
            constexpr int k = kc.value;
            if (k == 0) load_x(xr[0], 0, st);
            if (k == 0 && kPer > 1) load_x(xr[1], 1, st);
            if (k == 3) store_x(xr[0], 0, b);
            if (k == 3 && kPer > 2) load_x(xr[0], 2, st);
            if (k == 4 && kPer > 1) store_x(xr[1], 1, b);
            if (k == 4 && kPer > 3) load_x(xr[1], 3, st);
            if (k == 6 && kPer > 2) store_x(xr[0], 2, b);
            if (k == 7 && kPer > 3) store_x(xr[1], 3, b);
        },
        [&] {
#pragma unroll
            for (int j = 0; j < kPer; j++) {
                const int q = wave + kWaves * j, row = 16 * ((q >> 2) % MT) + 4 * (q & 3);
                if (found[j] == 0u) continue;
                uint32_t rows = 0u;
#pragma unroll
                for (int i = 0; i < 4; i++)
                    rows |= ((found[j] >> (16 * i)) & 0xFFFFu) != 0u && m0 + row + i < M ? 1u << i : 0u;
                if (lane == 0) atomicOr(&wide[row >> 5], rows << (row & 31));  // LDS atomic
            }
        });
    uint32_t any = 0u;
#pragma unroll
    for (int i = 0; i < (kTileM + 31) / 32; i++) any |= wide[i];
    if (__builtin_amdgcn_readfirstlane((int)any) != 0)
        kq_wide_rows<T, MT>(wide, acc, wp, st0, st1, nsb, lane, sb_of, [&](int row, int sb, int c, float (&v)[16]) {
            const int r = m0 + row;
            const v4u *const p = reinterpret_cast<const v4u *>(X + (int64_t)(r < M ? r : M - 1) * K + (int64_t)sb * kQK + 16 * c);
            const v4u a = p[0], b = p[1];
#pragma unroll
            for (int i = 0; i < 16; i++) {
                const uint32_t w = (i < 8 ? a : b)[(i >> 1) & 3];
                v[i] = __uint_as_float((i & 1) ? w & 0xFFFF0000u : w << 16);
            }
        });

    if constexpr (KW > 1) {
        f32x4 *const red = reinterpret_cast<f32x4 *>(lds[0]);
        if (kw > 0) {
#pragma unroll
            for (int mt = 0; mt < MT; mt++)
#pragma unroll
                for (int nt = 0; nt < 2; nt++) red[((wave * MT + mt) * 2 + nt) * 64 + lane] = acc[mt][nt];
        }
        __syncthreads();
        if (kw > 0) return;
#pragma unroll
        for (int k = 1; k < KW; k++)
#pragma unroll
            for (int mt = 0; mt < MT; mt++)
#pragma unroll
                for (int nt = 0; nt < 2; nt++) acc[mt][nt] += red[(((k * NW + nw) * MT + mt) * 2 + nt) * 64 + lane];
    }
    float *const out = split == 0 ? Y : part + (int64_t)(split - 1) * M * N;
#pragma unroll
    for (int mt = 0; mt < MT; mt++)
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const int m = m0 + 16 * mt + 4 * g + r;
#pragma unroll
            for (int nt = 0; nt < 2; nt++) {
                const int c = col0 + 16 * nt + n;
                if (m < M && c < N) out[(int64_t)m * N + c] = acc[mt][nt][r];
            }
        }
}

namespace {

// Fitted per type (gguf_gemm_plan.hpp).
constexpr GemmPlanCost kQ4KPlans[] = {
    {1, 1, 4, 2, 3.30f, 2.87f}, {1, 1, 8, 1, 2.70f, 3.17f}, {1, 2, 4, 1, 2.19f, 2.19f},
    {2, 2, 2, 2, 3.90f, 3.25f}, {2, 2, 4, 1, 2.98f, 3.31f}, {2, 4, 2, 1, 2.94f, 2.51f},
    {4, 4, 2, 1, 4.18f, 3.71f}, {4, 8, 1, 1, 3.77f, 2.96f}, {6, 8, 1, 1, 5.51f, 3.73f},
    {8, 8, 1, 1, 6.48f, 4.90f}};
constexpr GemmSplitCost kQ4KSplit = {2.88f, 0.179f};
constexpr GemmPlanCost kQ5KPlans[] = {
    {1, 1, 4, 2, 3.49f, 3.74f}, {1, 1, 8, 1, 2.65f, 4.14f}, {1, 2, 4, 1, 2.23f, 3.24f},
    {2, 2, 2, 2, 3.55f, 4.06f}, {2, 2, 4, 1, 2.88f, 4.32f}, {2, 4, 2, 1, 3.03f, 3.40f},
    {4, 4, 2, 1, 3.86f, 4.71f}, {4, 8, 1, 1, 3.64f, 3.69f}, {6, 8, 1, 1, 4.70f, 4.79f},
    {8, 8, 1, 1, 5.19f, 5.66f}};
constexpr GemmSplitCost kQ5KSplit = {2.85f, 0.218f};
constexpr GemmPlanCost kQ6KPlans[] = {
    {1, 1, 4, 2, 2.90f, 4.64f}, {1, 1, 8, 1, 2.64f, 5.33f}, {1, 2, 4, 1, 2.15f, 4.68f},
    {2, 2, 2, 2, 3.17f, 4.65f}, {2, 2, 4, 1, 2.92f, 5.39f}, {2, 4, 2, 1, 2.59f, 4.59f},
    {4, 4, 2, 1, 3.66f, 5.65f}, {4, 8, 1, 1, 3.57f, 5.04f}, {6, 8, 1, 1, 4.62f, 6.15f},
    {8, 8, 1, 1, 5.23f, 7.90f}};
constexpr GemmSplitCost kQ6KSplit = {2.97f, 0.203f};

GemmPlan kq_plan(int type_id, int M, int N, int K, size_t ws_bytes) {
    if (type_id == kQ4_K) return pick_gemm_plan(kQ4KPlans, kQ4KSplit, M, N, K, ws_bytes);
    if (type_id == kQ5_K) return pick_gemm_plan(kQ5KPlans, kQ5KSplit, M, N, K, ws_bytes);
    return pick_gemm_plan(kQ6KPlans, kQ6KSplit, M, N, K, ws_bytes);
}

template <int T, int MT, int NW, int KW>
void launch(unsigned grid, hipStream_t stream, const uint8_t *w, int64_t row_bytes, const uint16_t *x, float *y,
            int M, int N, int K, int S, float *part) {
    hipLaunchKernelGGL((gemm_kq_kernel<T, MT, NW, KW>), dim3(grid), dim3(64 * NW * KW), 0, stream, w, row_bytes, x, y,
                       M, N, K, S, part);
}

template <int T, class... A>
bool launch_plan(const GemmPlan &p, A... a) {
    const int key = 100 * p.mt + 10 * p.nw + p.kw;
    switch (key) {
    case 114: launch<T, 1, 1, 4>(a...); break;
    case 118: launch<T, 1, 1, 8>(a...); break;
    case 124: launch<T, 1, 2, 4>(a...); break;
    case 222: launch<T, 2, 2, 2>(a...); break;
    case 224: launch<T, 2, 2, 4>(a...); break;
    case 242: launch<T, 2, 4, 2>(a...); break;
    case 442: launch<T, 4, 4, 2>(a...); break;
    case 481: launch<T, 4, 8, 1>(a...); break;
    case 681: launch<T, 6, 8, 1>(a...); break;
    case 881: launch<T, 8, 8, 1>(a...); break;
    default: return false;
    }
    return true;
}

}  // namespace

bool kq_gemm_supported(int type_id, int64_t row_bytes, int N, int K, const void *w, const void *x) {
    // (Q4_K: 128 rows of X lie within the 2^31 bytes of a buffer descriptor)
    return (type_id == kQ4_K || type_id == kQ5_K || type_id == kQ6_K) && K > 0 && K % kQK == 0 && N > 0 &&
           (type_id != kQ4_K || K < 1 << 23) &&
           ((reinterpret_cast<uintptr_t>(w) | (uintptr_t)row_bytes) & 1u) == 0 &&
           (reinterpret_cast<uintptr_t>(x) & 15u) == 0;
}

size_t kq_gemm_workspace_bytes(int type_id, int M, int N, int K) {
    if (!gemm_may_split(type_id, M, N, K)) return 0;
    return gemm_plan_bytes(kq_plan(type_id, M, N, K, kGemmMaxSplitBytes), M, N);
}

void kq_gemm_plan(int type_id, int M, int N, int K, int32_t (&plan)[4]) {
    const bool split = gemm_may_split(type_id, M, N, K) && ((int64_t)M * N) % 4 == 0;
    const GemmPlan p = kq_plan(type_id, M, N, K, split ? kGemmMaxSplitBytes : 0);
    plan[0] = p.mt;
    plan[1] = p.nw;
    plan[2] = p.kw;
    plan[3] = p.splits;
}

hipError_t launch_kq_gemm(int type_id, const uint8_t *w, int64_t row_bytes, const uint16_t *x, float *y, int M, int N,
                          int K, hipStream_t stream, float *workspace, size_t workspace_bytes) {
    const bool split = workspace != nullptr && gemm_may_split(type_id, M, N, K) && ((int64_t)M * N) % 4 == 0 &&
                       ((reinterpret_cast<uintptr_t>(workspace) | reinterpret_cast<uintptr_t>(y)) & 15u) == 0;
    const GemmPlan p = kq_plan(type_id, M, N, K, split ? workspace_bytes : 0);
    const unsigned grid =
        (unsigned)(((M + 16 * p.mt - 1) / (16 * p.mt)) * ((N + 32 * p.nw - 1) / (32 * p.nw)) * p.splits);
    bool ok;
    if (type_id == kQ4_K) ok = launch_plan<kQ4_K>(p, grid, stream, w, row_bytes, x, y, M, N, K, p.splits, workspace);
    else if (type_id == kQ5_K) ok = launch_plan<kQ5_K>(p, grid, stream, w, row_bytes, x, y, M, N, K, p.splits, workspace);
    else ok = launch_plan<kQ6_K>(p, grid, stream, w, row_bytes, x, y, M, N, K, p.splits, workspace);
    if (!ok) return hipErrorInvalidValue;
    if (p.splits > 1) return launch_gemm_reduce(workspace, p.splits, (int64_t)M * N, y, stream);
    return hipGetLastError();
}

}  // namespace gollek
