// gguf_moe_gemm.hip -- grouped MoE expert FFN for many routes per expert
// (prefill): Q4_K, Q5_K or Q6_K experts on the fp16 matrix cores
// (gguf_kq_f16.hpp).
//
// Semantics as gguf_moe.hip (MoeForwardPass.java:217-240, :461-472; swigluFfn
// DirectForwardFfnService.java:40-61).  Up to 16 MT routes of an expert are
// the rows of one GEMM tile, so its weights are read and widened once for all
// of them instead of once per four routes.
//
// fp32 vectors are two fp16 digits: with a row's superblock scaled to a
// maximum in [2^14, 2^15), v = hi + lo leaves an error below 2^-23 of v or 2^-39
// of the maximum (the two-launch passes keep 2^-22 of it; against the fp32 row
// kernels the roundings of the products weigh more: 4.5e-7 of error against
// 7e-7); both digits contract against the same exact weight operand into one
// fp32 accumulator.
// They are built once per vector ("records") by a kernel of its own, x's into
// the workspace's ypair region (free until the down pass), h's in place.
// Superblocks of too wide a range and those with an infinity (kq_wide) stay
// fp32, marked by a negative scale, and the rows that hold one are computed
// again from the packed weights -- on the shapes that only the fp32 row kernels
// take otherwise.  Where the two-launch passes do, x and h were digits of 22 bits
// already, and h may well be of that kind (gates far below 0: e^-|g| over many
// powers of two; 256 tokens of random weights 154 us without, 187 with).
//
// What bounds it: a workgroup's stage is short (34 MFMAs a wave at one row
// tile), so its loads' latency shows; small tiles keep several workgroups on
// a CU.  128 experts x 768, hidden 2048, Q4_K gate / up, Q6_K down, 256 tokens x
// top-8: 714 us on the passes of gguf_moe_mfma.hip, 176 here (the launches beside
// the two GEMMs 25 us; the weights are 391 MB); 32 x 1280, hidden 2816, 100 tokens
// x top-4: 918 us on the row kernels, 109 here.
//
// Launches: routing (a list of (expert, first route) items of at most 16 MT
// routes) with x's records, gate/up (h), h records, down (a row per route), combine
// in route order.
#include "gguf_dot4.hpp"
#include "gguf_kernels.hpp"
#include "gguf_kq_f16.hpp"
#include "gguf_moe_route.hpp"

namespace gollek {

using namespace kqf;

namespace {

// Tail of a (row, superblock) record: the min pieces and the inverse scale.
constexpr int kTailBytes = 64;

}  // namespace

namespace {

// One row's superblock, fp32 -> record (16 lanes of a wave, 16 columns each):
// rec (row, superblock) 1024 bytes, per half and digit 16 pieces (KqUnit's
// order, not swizzled); mins 64 bytes; scales one float.  A wide superblock's
// rec is its 256 floats and its scale negative (mins not written).  The lanes
// have read their columns before they write (rec may be v itself).
template <int T>
__device__ __forceinline__ void record_row(const float *v, int64_t r, int sb, int K, int keep_wide, uint8_t *rec,
                                           uint8_t *__restrict__ mins, float *__restrict__ scales) {
    const int n = (int)threadIdx.x & 15;
    const int64_t rs = r * (K / kQK) + sb;
    const f32x4 *const src = reinterpret_cast<const f32x4 *>(v + r * K + kQK * sb + 16 * n);
    f32x4 x[4];
#pragma unroll
    for (int i = 0; i < 4; i++) x[i] = src[i];
    float mx = 0.0f;
#pragma unroll
    for (int i = 0; i < 16; i++) mx = fmaxf(mx, fabsf(x[i >> 2][i & 3]));
    const float lane_mx = mx;
    mx = row_max16(mx);
    float s, inv, t = 0.0f;
    kq_row_scale(mx, s, inv);
    uint8_t *const dst = rec + rs * 1024;
    const uint64_t found = kq_wide(lane_mx, mx, inv);
    if (keep_wide && __popc((uint32_t)(found >> (threadIdx.x & 48u)) & 0xFFFFu) >= kWideRuns) {  // the row's lanes alike
#pragma unroll
        for (int i = 0; i < 4; i++) reinterpret_cast<f32x4 *>(dst + 64 * n)[i] = x[i];
        if (n == 0) scales[rs] = -inv;
        return;
    }
    int g, kk[2];
    kq_place<T>(n, g, kk[0], kk[1]);
#pragma unroll
    for (int h = 0; h < 2; h++) {
        uint32_t f[2][4];
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const int e = 8 * h + 4 * (j >> 1) + (j & 1);
            const float a = x[e >> 2][e & 3] * s, b = x[(e + 2) >> 2][(e + 2) & 3] * s;
            const f16x2 hi = {(_Float16)a, (_Float16)b};
            const f16x2 lo = {(_Float16)(a - (float)hi[0]), (_Float16)(b - (float)hi[1])};
            f[0][j] = as_u(hi);
            f[1][j] = as_u(lo);
            t += a + b;
        }
#pragma unroll
        for (int d = 0; d < 2; d++)
            *reinterpret_cast<f16x8 *>(dst + 512 * (kk[h] >> 2) + 256 * d + 16 * (4 * (kk[h] & 3) + g)) = as_h8(f[d]);
    }
    if constexpr (KqOperand<T, true>::kMins) {
        t += kq_dpp<0xB1>(t);  // the sub-block's other 16 columns
        *reinterpret_cast<uint2 *>(mins + rs * kTailBytes + 16 * (n >> 2) + 8 * ((n >> 1) & 1)) =
            kq_min_digits(t * 0x1p-6f);
    }
    if (n == 0) scales[rs] = inv;
}

}  // namespace

// Records of `rows` rows, 16 rows and a superblock a workgroup.
template <int T>
__global__ __launch_bounds__(256) void moe_records_kernel(const float *v, int rows, int K, int keep_wide, uint8_t *rec,
                                                          uint8_t *__restrict__ mins, float *__restrict__ scales) {
    const int r = 16 * (int)blockIdx.y + (int)(threadIdx.x >> 4);
    if (r < rows) record_row<T>(v, r, (int)blockIdx.x, K, keep_wide, rec, mins, scales);  // whole rows of 16 lanes
}

// The first launch: workgroup 0 routes, the others build x's records (64 rows'
// superblocks each), which do not depend on it.  (As two launches 5 us more.)
template <int T>
__global__ __launch_bounds__(kRouteThreads) void moe_front_kernel(const int32_t *__restrict__ ids,
                                                                  const float *__restrict__ wts, int P, int E,
                                                                  int group, int chunks, int keys_in_lds,
                                                                  int32_t *__restrict__ meta,
                                                                  int2 *__restrict__ items, const float *x, int rows,
                                                                  int K, int keep_wide, uint8_t *rec,
                                                                  uint8_t *__restrict__ mins,
                                                                  float *__restrict__ scales) {
    extern __shared__ int32_t sh[];
    if (blockIdx.x == 0) {
        moe_route(ids, wts, P, E, group, chunks, keys_in_lds, meta, items, sh);
        return;
    }
    const int nsb = K / kQK;
    const int64_t i = (int64_t)(blockIdx.x - 1) * (kRouteThreads / 16) + (int)(threadIdx.x >> 4);
    if (i < (int64_t)rows * nsb) record_row<T>(x, i / nsb, (int)(i % nsb), K, keep_wide, rec, mins, scales);
}

namespace {

// Columns 16 c .. + 15 of a record.
template <int T>
__device__ __forceinline__ void record_columns(const uint8_t *rec, float scale, int c, float (&v)[16]) {
    if (scale < 0.0f) {
        const f32x4 *const p = reinterpret_cast<const f32x4 *>(rec + 64 * c);
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const f32x4 x = p[i];
#pragma unroll
            for (int j = 0; j < 4; j++) v[4 * i + j] = x[j];
        }
        return;
    }
    int g, kk[2];
    kq_place<T>(c, g, kk[0], kk[1]);
#pragma unroll
    for (int h = 0; h < 2; h++) {
        const uint8_t *const p = rec + 512 * (kk[h] >> 2) + 16 * (4 * (kk[h] & 3) + g);
        const f16x8 hi = *reinterpret_cast<const f16x8 *>(p), lo = *reinterpret_cast<const f16x8 *>(p + 256);
#pragma unroll
        for (int e = 0; e < 8; e++) {  // slot e holds column 0, 2, 1, 3, 4, 6, 5, 7
            const int col = (e & 4) | ((e & 1) << 1) | ((e >> 1) & 1);
            v[8 * h + col] = ((float)hi[e] + (float)lo[e]) * scale;
        }
    }
}

// One item's tile: MT row tiles (cnt routes) x 32 NW weight rows.
template <int T, int MT, int NW, bool GATED>
__device__ __forceinline__ void moe_item(const uint8_t *const (&wp)[2], int nsb, const uint8_t *__restrict__ rec,
                                         const uint8_t *__restrict__ mins, const float *__restrict__ scales,
                                         const int *rows, const int *routes, int cnt, uint8_t *lds,
                                         uint32_t *wide_rows, float *out, int out_stride, int col) {
    using U = KqUnit<2>;
    constexpr int kThreads = 64 * NW;
    constexpr int kBatch = 4, kLoads = 1024 * MT / kThreads, kBatches = (kLoads + kBatch - 1) / kBatch;
    static_assert(64 * MT <= kThreads, "a min piece per thread");
    const int tid = (int)threadIdx.x, lane = tid & 63, n = lane & 15, g = lane >> 4;
    f32x4 acc[MT][2];
#pragma unroll
    for (int mt = 0; mt < MT; mt++)
#pragma unroll
        for (int nt = 0; nt < 2; nt++) acc[mt][nt] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};

    // A load takes one row's record of the stage per wave (64 pieces).
    v4u st[kBatch], tail;
    float sc = 0.0f;
    bool wide = false;  // row tid has a wide superblock
    auto load = [&](int bt, int sb) {
#pragma unroll
        for (int j = 0; j < kBatch; j++) {
            const int c = (bt * kBatch + j) * kThreads + tid;
            if (bt * kBatch + j < kLoads)
                st[j] = *reinterpret_cast<const v4u *>(rec + ((int64_t)rows[c >> 6] * nsb + sb) * 1024 + 16 * (c & 63));
        }
    };
    auto store = [&](int bt, int b) {
#pragma unroll
        for (int j = 0; j < kBatch; j++) {
            const int c = (bt * kBatch + j) * kThreads + tid, r = c >> 6, p = c & 63;
            if (bt * kBatch + j < kLoads)
                *reinterpret_cast<v4u *>(lds + (b * MT + (r >> 4)) * U::kBytes + U::kHalf * (p >> 5) +
                                         U::kDigit * ((p >> 4) & 1) + 256 * (r & 15) + 16 * ((p & 15) ^ (r & 15))) = st[j];
        }
    };
    auto load_tail = [&](int sb) {
        if constexpr (KqOperand<T, true>::kMins)
            if (tid < 64 * MT)
                tail = *reinterpret_cast<const v4u *>(mins + ((int64_t)rows[tid >> 2] * nsb + sb) * kTailBytes + 16 * (tid & 3));
        if (tid < 16 * MT) sc = scales[(int64_t)rows[tid] * nsb + sb];
    };
    auto store_tail = [&](int b) {
        if constexpr (KqOperand<T, true>::kMins)
            if (tid < 64 * MT)
                *reinterpret_cast<v4u *>(lds + (b * MT + (tid >> 6)) * U::kBytes + U::kMins + 16 * (tid & 63)) = tail;
        wide |= sc < 0.0f;
        if (tid < 16 * MT)
            *reinterpret_cast<float *>(lds + (b * MT + (tid >> 4)) * U::kBytes + U::kScales + 4 * (tid & 15)) = sc;
    };
    kq_stages<T, MT, 2, true, true>(acc, wp, lds, MT * U::kBytes, 0, nsb, nsb, lane, [](int st) { return st; },
                        [&] {  // (requesting W before x is in LDS changed nothing here)
                            load_tail(0);
#pragma unroll
                            for (int bt = 0; bt < kBatches; bt++) {
                                load(bt, 0);
                                store(bt, 0);
                            }
                            store_tail(0);
                            __syncthreads();
                        },
                        [] {},
                        [&](auto kc, int sb, int b) {
                            constexpr int k = kc.value, per = 8 / kBatches;
                            if constexpr (k == 0) load_tail(sb);
                            if constexpr (k > 0 && k % per == 0) store(k / per - 1, b);
                            if constexpr (k % per == 0) load(k / per, sb);
                            if constexpr (k == 7) {
                                store(kBatches - 1, b);
                                store_tail(b);
                            }
                        },
                        [&] {  // (rows past cnt repeat the last route's)
                            const uint32_t found = (uint32_t)__builtin_amdgcn_ballot_w64(wide && tid < cnt);
                            if (tid == 0) *wide_rows = found;
                        });
    if (__builtin_amdgcn_readfirstlane((int)*wide_rows) != 0)
        kq_wide_rows<T, MT>(wide_rows, acc, wp, 0, nsb, nsb, lane, [](int st) { return st; },
                            [&](int row, int sb, int c, float (&v)[16]) {
                                const int64_t rs = (int64_t)rows[row] * nsb + sb;
                                record_columns<T>(rec + rs * 1024, scales[rs], c, v);
                            });
#pragma unroll
    for (int mt = 0; mt < MT; mt++)
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const int m = 16 * mt + 4 * g + r;
            if (m >= cnt) continue;
            float *const dst = out + (int64_t)routes[m] * out_stride + col + n;
            if constexpr (GATED) {
                const float a = acc[mt][0][r];
                dst[0] = a / (1.0f + expf(-a)) * acc[mt][1][r];  // silu(gate) * up
            } else {
                dst[0] = acc[mt][0][r];
                dst[16] = acc[mt][1][r];
            }
        }
}

}  // namespace

// One workgroup: an item (expert, up to 16 MTMAX of its routes) and 32 NW
// weight rows: GATED 16 NW gate rows and the same up rows, else down rows.
// Items of fewer row tiles take the loop for their count.
template <int T, int MTMAX, int NW, bool GATED>
__global__ __launch_bounds__(64 * NW) void moe_gemm_kernel(const uint8_t *__restrict__ w0,
                                                           const uint8_t *__restrict__ w1, int rows_e, int K,
                                                           const uint8_t *__restrict__ rec,
                                                           const uint8_t *__restrict__ mins,
                                                           const float *__restrict__ scales, int per_record,
                                                           const int2 *__restrict__ items,
                                                           const int32_t *__restrict__ nitems,
                                                           const int32_t *__restrict__ offsets,
                                                           const int32_t *__restrict__ pairs, float *out) {
    constexpr int kCols = (GATED ? 16 : 32) * NW;
    __shared__ __attribute__((aligned(16))) uint8_t lds[2 * MTMAX * KqUnit<2>::kBytes];
    __shared__ int rows[16 * MTMAX], routes[16 * MTMAX];
    __shared__ uint32_t wide_rows;  // one bit a row
    const int slices = rows_e / kCols, item = (int)blockIdx.x / slices, slice = (int)blockIdx.x - item * slices;
    if (item >= *nitems) return;
    const int2 it = items[item];
    const int left = offsets[it.x + 1] - it.y, cnt = left < 16 * MTMAX ? left : 16 * MTMAX;
    const int tid = (int)threadIdx.x, n = tid & 15, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int nsb = K / kQK;
    const int64_t row_bytes = (int64_t)nsb * kq_block_bytes<T>();
    const int col = slice * kCols + (GATED ? 16 : 32) * wave;
    const uint8_t *wp[2];
    const int64_t first = (int64_t)it.x * rows_e + col + n;
    wp[0] = w0 + first * row_bytes;
    wp[1] = GATED ? w1 + first * row_bytes : w0 + (first + 16) * row_bytes;
    if (tid < 16 * MTMAX) {
        const int p = pairs[it.y + (tid < cnt ? tid : cnt - 1)];
        routes[tid] = p;
        rows[tid] = p / per_record;
    }
    __syncthreads();
    const int out_stride = rows_e;
    if constexpr (MTMAX == 2) {
        if (cnt > 16) {
            moe_item<T, 2, NW, GATED>(wp, nsb, rec, mins, scales, rows, routes, cnt, lds, &wide_rows, out, out_stride, col);
            return;
        }
    }
    moe_item<T, 1, NW, GATED>(wp, nsb, rec, mins, scales, rows, routes, cnt, lds, &wide_rows, out, out_stride, col);
}

namespace {

// Records' tails and the item list in the workspace's xdig / hdig regions.
struct RecordTails {
    size_t mins, scales, end;  // byte offsets
};
RecordTails tails_at(size_t at, int64_t rows, int nsb) {
    RecordTails t;
    t.mins = at;
    t.scales = t.mins + (size_t)rows * nsb * kTailBytes;
    t.end = t.scales + (size_t)rows * nsb * 4;
    return t;
}

// Row tiles of an item: one keeps 16-row items' LDS small (four workgroups on
// a CU instead of two), two read an expert's weights once for up to 32
// routes.  128 experts x 768 (hidden 2048, Q4_K): 8 routes per expert 125 us
// with one, 136 with two; 16 routes per expert 173 / 168; 64 x 1024, 24
// routes: 129 / 117 us.
int item_tiles(int64_t P, int E) { return P >= 10 * (int64_t)E ? 2 : 1; }

int64_t max_items(int64_t P, int E, int group) { return (P < E ? P : E) + P / group; }

// Waves of a workgroup.  Eight stage x once for twice the weight rows, but one
// such workgroup fills a CU: from two rounds over the CUs, by the items to be
// expected (half a tile more than the routes fill, per expert).  128 x 768, 256
// tokens x top-8, three rounds: 209 us with four, 194 with eight; 32 x 1280,
// 100 tokens x top-4, 1.25 rounds: 156 / 184 us.
bool wide_groups(int64_t P, int E, int mt, int rows_e, int cols) {
    return (P / (16 * mt) + E / 2) * (rows_e / cols) >= 2 * (int64_t)device_cus();
}

template <int T, int MT, int NW, bool GATED, class... A>
hipError_t launch_groups(unsigned items, int rows_e, hipStream_t stream, A... a) {
    hipLaunchKernelGGL((moe_gemm_kernel<T, MT, NW, GATED>), dim3(items * (unsigned)(rows_e / ((GATED ? 16 : 32) * NW))),
                       dim3(64 * NW), 0, stream, a...);
    return hipGetLastError();
}

template <int T, bool GATED>
hipError_t launch_pass(int mt, int64_t P, int E, unsigned items, const uint8_t *w0, const uint8_t *w1, int rows_e,
                       int K, const uint8_t *rec, const uint8_t *mins, const float *scales, int per_record,
                       const int2 *list, const int32_t *nitems, const int32_t *offsets, const int32_t *pairs,
                       float *out, hipStream_t stream) {
    auto run = [&](auto launch) {
        return launch(items, rows_e, stream, w0, w1, rows_e, K, rec, mins, scales, per_record, list, nitems, offsets,
                      pairs, out);
    };
    const bool wide = wide_groups(P, E, mt, rows_e, (GATED ? 16 : 32) * 8);
    if (mt == 1)
        return wide ? run([](auto... a) { return launch_groups<T, 1, 8, GATED>(a...); })
                    : run([](auto... a) { return launch_groups<T, 1, 4, GATED>(a...); });
    return wide ? run([](auto... a) { return launch_groups<T, 2, 8, GATED>(a...); })
                : run([](auto... a) { return launch_groups<T, 2, 4, GATED>(a...); });
}

template <bool GATED, class... A>
hipError_t launch_pass_type(int type, A... a) {
    if (type == kQ4_K) return launch_pass<kQ4_K, GATED>(a...);
    if (type == kQ5_K) return launch_pass<kQ5_K, GATED>(a...);
    return launch_pass<kQ6_K, GATED>(a...);
}

hipError_t launch_records(int type, const float *v, int64_t rows, int K, bool keep_wide, uint8_t *rec, uint8_t *mins,
                          float *scales, hipStream_t stream) {
    const dim3 grid((unsigned)(K / kQK), (unsigned)((rows + 15) / 16));
    if (type == kQ6_K)
        hipLaunchKernelGGL(moe_records_kernel<kQ6_K>, grid, dim3(256), 0, stream, v, (int)rows, K,
                           (int)keep_wide, rec, mins, scales);
    else
        hipLaunchKernelGGL(moe_records_kernel<kQ4_K>, grid, dim3(256), 0, stream, v, (int)rows, K,
                           (int)keep_wide, rec, mins, scales);
    return hipGetLastError();
}

bool kq_type(int t) { return t == kQ4_K || t == kQ5_K || t == kQ6_K; }

}  // namespace

bool moe_gemm_supported(int gate_type, int up_type, int down_type, int E, int H, int I, int T, int top_k,
                        const uint8_t *gate, const uint8_t *up, const uint8_t *down, const float *x) {
    if (gate_type != up_type || !kq_type(gate_type) || !kq_type(down_type)) return false;
    if (H % kQK != 0 || I % kQK != 0 || H < kQK || I < kQK || T < 1 || top_k < 1) return false;
    if (((reinterpret_cast<uintptr_t>(gate) | reinterpret_cast<uintptr_t>(up) | reinterpret_cast<uintptr_t>(down)) & 1u) != 0 ||
        (reinterpret_cast<uintptr_t>(x) & 15u) != 0)
        return false;
    const int64_t P = (int64_t)T * top_k;
    const MoeLayout L = moe_layout(T, top_k, H, I, E);
    const int64_t items = max_items(P, E, 16 * item_tiles(P, E));
    const RecordTails xt = tails_at(L.xdig, T, H / kQK);
    return (xt.end + 15) / 16 * 16 + (size_t)items * 8 <= L.h && tails_at(L.hdig, P, I / kQK).end <= L.ypair &&
           (P + 15) / 16 <= 65535 &&
           // threads of the passes: four a gate row and item, two a down row
           items * (4 * (int64_t)I > 2 * (int64_t)H ? 4 * (int64_t)I : 2 * (int64_t)H) < ((int64_t)1 << 32);
}

hipError_t launch_moe_gemm(int gate_type, int down_type, const uint8_t *gate, const uint8_t *up, const uint8_t *down,
                           int E, int H, int I, const float *x, const int32_t *ids, const float *wts, int T,
                           int top_k, bool keep_wide, float *out, uint8_t *ws, hipStream_t stream) {
    const MoeLayout L = moe_layout(T, top_k, H, I, E);
    const int P = T * top_k, mt = item_tiles(P, E);
    int32_t *meta = reinterpret_cast<int32_t *>(ws + L.meta);
    const RecordTails xt = tails_at(L.xdig, T, H / kQK), ht = tails_at(L.hdig, P, I / kQK);
    int2 *list = reinterpret_cast<int2 *>(ws + (xt.end + 15) / 16 * 16);
    const int32_t *offsets = meta + E, *pairs = meta + 2 * E + 1, *nitems = pairs + P + E + 1;
    const unsigned items = (unsigned)max_items(P, E, 16 * mt);
    uint8_t *xrec = ws + L.ypair, *hrec = ws + L.h;
    float *h = reinterpret_cast<float *>(hrec), *ypair = reinterpret_cast<float *>(ws + L.ypair);
    const MoeRoutePlan rp = moe_route_plan(P, E);
    const int64_t xrows = (int64_t)T * (H / kQK);
    const dim3 fgrid((unsigned)(1 + (xrows + kRouteThreads / 16 - 1) / (kRouteThreads / 16)));
    auto front = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, fgrid, dim3(kRouteThreads), rp.lds_bytes, stream, ids, wts, P, E, 16 * mt,
                           rp.chunks, rp.keys_in_lds, meta, list, x, T, H, (int)keep_wide, xrec, ws + xt.mins,
                           reinterpret_cast<float *>(ws + xt.scales));
    };
    gate_type == kQ6_K ? front(&moe_front_kernel<kQ6_K>) : front(&moe_front_kernel<kQ4_K>);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    e = launch_pass_type<true>(gate_type, mt, (int64_t)P, E, items, gate, up, I, H, xrec, ws + xt.mins,
                               reinterpret_cast<const float *>(ws + xt.scales), top_k, list, nitems, offsets, pairs, h,
                               stream);
    if (e != hipSuccess) return e;
    e = launch_records(down_type, h, P, I, keep_wide, hrec, ws + ht.mins, reinterpret_cast<float *>(ws + ht.scales), stream);
    if (e != hipSuccess) return e;
    e = launch_pass_type<false>(down_type, mt, (int64_t)P, E, items, down, down, H, I, hrec, ws + ht.mins,
                                reinterpret_cast<const float *>(ws + ht.scales), 1, list, nitems, offsets, pairs,
                                ypair, stream);
    if (e != hipSuccess) return e;
    return launch_moe_combine(ids, wts, ypair, T, top_k, H, E, out, stream);
}

}  // namespace gollek
