// gguf_moe_route.hpp -- MoE routing on one workgroup (gguf_moe.hip,
// gguf_moe_gemm.hip).
#pragma once

#include "gguf_kernels.hpp"

namespace gollek {

constexpr int kRouteThreads = 1024;

// Launch parameters of the routing: a chunk a wave of the workgroup while their
// counters fit 32 KB (one for few routes, whose serial scatter is shorter than
// the larger workgroup's start), and the routes' keys in LDS for the scatter
// while everything fits the default 64 KB (it otherwise reloads them, one
// round trip per 64).
struct MoeRoutePlan {
    int threads, chunks, keys_in_lds;
    size_t lds_bytes;
};
inline MoeRoutePlan moe_route_plan(int P, int E) {
    MoeRoutePlan p;
    p.threads = P <= 512 ? 256 : kRouteThreads;
    p.chunks = P > 512 && 16 * (size_t)E * sizeof(int32_t) <= 32768 ? 16 : 1;
    const size_t base = (size_t)(1 + p.chunks) * (size_t)E * sizeof(int32_t);
    p.keys_in_lds = base + (size_t)P * sizeof(int32_t) <= 65536 ? 1 : 0;
    p.lds_bytes = base + (p.keys_in_lds ? (size_t)P * sizeof(int32_t) : 0);
    return p;
}

// Routing on one workgroup: per-expert counts of the valid routes (expert id
// in range, weight != 0; MFP:222), their offsets, the route list stably
// sorted by expert, the used experts in expert order, and (group > 0) the
// items of the grouped GEMM, (expert, first route in that order) for every
// `group` routes of an expert.  Wave 0 scans in chunks of 64 with DPP-free
// shuffles; the stable scatter ranks equal keys within a chunk by ballots.
// The routes are cut into `chunks` runs, one a wave (1: all of them in wave
// 0's scatter): each counts its own keys, so the scatters run side by side
// (2048 routes: 23 us in one wave, 6.6 us in 16).
// Called by all threads of the workgroup (at least 64 a chunk); sh: the plan's LDS
// bytes, cnt[E], run[chunks][E], then (keys_in_lds) key[P].
__device__ inline void moe_route(const int32_t *__restrict__ ids, const float *__restrict__ wts, int P, int E,
                                 int group, int chunks, int keys_in_lds, int32_t *__restrict__ meta,
                                 int2 *__restrict__ items, int32_t *sh) {
    int32_t *cnt = sh, *run = sh + E, *keys = run + chunks * E;
    int32_t *counts = meta, *offsets = meta + E, *pairs = meta + 2 * E + 1;
    int32_t *used = pairs + P, *nused = used + E;
    int32_t *nitems = nused + 1;
    const int tid = (int)threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int per = ((P + chunks - 1) / chunks + 63) / 64 * 64;  // routes of a chunk
    for (int i = tid; i < chunks * E; i += (int)blockDim.x) run[i] = 0;
    __syncthreads();
    for (int p = tid; p < P; p += (int)blockDim.x) {
        const int e = ids[p];
        const bool valid = e >= 0 && e < E && wts[p] != 0.0f;
        if (valid) atomicAdd(&run[p / per * E + e], 1);  // LDS atomic
        if (keys_in_lds) keys[p] = valid ? e : -1;
    }
    __syncthreads();
    // (one chunk: its counts are the experts', and wave 0 goes on alone; with the
    // barriers below the row passes of a token took 0.17 us more, 17.3 in all)
    if (chunks > 1) {
        for (int e = tid; e < E; e += (int)blockDim.x) {
            int c = 0;
            for (int k = 0; k < chunks; k++) {
                const int n = run[k * E + e];
                run[k * E + e] = c;
                c += n;
            }
            cnt[e] = c;
        }
        __syncthreads();
    }
    const uint64_t below = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
    if (tid < 64) {
        int carry = 0, ucount = 0, icarry = 0;
        for (int base = 0; base < E; base += 64) {
            const int e = base + lane;
            const int c = e < E ? (chunks > 1 ? cnt[e] : run[e]) : 0;
            const int groups = group > 0 ? (c + group - 1) / group : 0;
            int a = c, b = groups;
            // inclusive scans over the 64 lanes
            for (int d = 1; d < 64; d <<= 1) {
                const int ta = __shfl_up(a, d, 64), tb = __shfl_up(b, d, 64);
                if (lane >= d) {
                    a += ta;
                    b += tb;
                }
            }
            const uint64_t ub = __ballot(c > 0);
            if (e < E) {
                offsets[e] = carry + a - c;
                counts[e] = c;
                cnt[e] = carry + a - c;
                if (chunks == 1) run[e] = 0;
            }
            if (c > 0) used[ucount + __popcll(ub & below)] = e;
            for (int i = 0; i < groups; i++) items[icarry + b - groups + i] = make_int2(e, carry + a - c + group * i);
            carry += __shfl(a, 63, 64);
            icarry += __shfl(b, 63, 64);
            ucount += __popcll(ub);
        }
        if (lane == 0) {
            offsets[E] = carry;
            *nused = ucount;
            *nitems = icarry;
        }
    }
    if (chunks > 1) __syncthreads();
    // Stable scatter, 64 routes at a time in route order: a route's slot is its
    // expert's offset, plus the routes of it in earlier chunks and rounds, plus
    // its rank among the round's equal keys.
    if (wave >= chunks) return;
    int32_t *const mine = run + wave * E;
    int bits = 1;
    while ((1 << bits) <= E) bits++;
    const int end = (wave + 1) * per < P ? (wave + 1) * per : P;
    for (int base = wave * per; base < end; base += 64) {
        const int p = base + lane;
        int key = -1;
        if (p < end) {
            if (keys_in_lds) {
                key = keys[p];
            } else {
                const int e = ids[p];
                if (e >= 0 && e < E && wts[p] != 0.0f) key = e;
            }
        }
        const uint32_t k1 = (uint32_t)(key + 1);
        uint64_t same = __ballot(true);
        for (int bt = 0; bt < bits; bt++) {
            const uint64_t v = __ballot((k1 >> bt) & 1u);
            same &= ((k1 >> bt) & 1u) ? v : ~v;
        }
        const int rank = __popcll(same & below);
        const int r0 = key >= 0 ? mine[key] : 0;  // read by all lanes before any update
        if (key >= 0) pairs[cnt[key] + r0 + rank] = p;
        const bool last = (same >> lane) == 1ull;  // highest lane of its key
        if (key >= 0 && last) mine[key] = r0 + __popcll(same);
    }
}

}  // namespace gollek
