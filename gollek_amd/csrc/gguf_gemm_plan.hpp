// gguf_gemm_plan.hpp -- tile and split choice of the register-widening GEMM
// (gguf_kq_gemm.hip).
//
// A tile is 16 mt rows of X by 32 nw rows of W on nw * kw waves, its stages kw
// chunks of 256 columns.  The time of a launch is modelled as the rounds of
// workgroups over the CUs (of the 256-column tiles by whole rounds, of the others
// half of it and half by the mean, since there a last round that is nearly empty
// runs faster) times a tile's start and end and its stages, plus, for K cut into S
// parts, the reduction launch.  (256 columns, Q4_K, N = 11008, K = 4096: 1.34 rounds
// of 64 rows 100 us, one round of 128 rows 85; 3.02 rounds of 96 rows at M = 1672
// 264, 2.35 of 128 254.)  The
// constants are fitted to all plans' times over M = 5 .. 2048 and twelve N x K
// (177 shapes a type): the plan picked is within 1 % of the fastest on average,
// one shape of a type at most 19 to 44 %.
#pragma once

#include <cstddef>

#include "gguf_kernels.hpp"

namespace gollek {

struct GemmPlan {
    int mt, nw, kw, splits;
};
struct GemmPlanCost {
    int mt, nw, kw;
    int per_cu;        // workgroups of a CU at a time
    float tile_us;     // a tile's start and end
    float stage_us;    // a stage
};
// The reduction of a split launch: its start, and per MB moved.
struct GemmSplitCost {
    float launch_us, mb_us;
};

// A workgroup's time alone on its CU, of that beside others.
constexpr double kGemmAlone = 0.7;

constexpr size_t kGemmMaxSplitBytes = (size_t)16 << 20;  // the static scratch of the no-allocation entry

// The fastest plan for Y[M, N] with K columns and `ws_bytes` for split-K
// partials (0: unsplit).
template <int PLANS>
GemmPlan pick_gemm_plan(const GemmPlanCost (&plans)[PLANS], GemmSplitCost split, int M, int N, int K,
                        size_t ws_bytes) {
    GemmPlan best{0, 0, 0, 1};
    double best_us = 0.0;
    const double cus = device_cus();
    const size_t mn = (size_t)M * N * sizeof(float);
    if (ws_bytes > kGemmMaxSplitBytes) ws_bytes = kGemmMaxSplitBytes;
    for (const GemmPlanCost &p : plans) {
        const long tiles = (long)((M + 16 * p.mt - 1) / (16 * p.mt)) * ((N + 32 * p.nw - 1) / (32 * p.nw));
        const int stages = ((K + 255) / 256 + p.kw - 1) / p.kw;
        for (int S = 1; S <= 8 && S <= stages && (S == 1 || (size_t)(S - 1) * mn <= ws_bytes); S++) {
            const double r = (double)tiles * S / (cus * p.per_cu);
            const double whole = (double)(long)(r + 0.999999);
            const double rounds = p.nw == 8 ? whole : 0.5 * whole + 0.5 * (r > 1.0 ? r : 1.0);
            double us = rounds * (p.tile_us + p.stage_us * ((stages + S - 1) / S));
            if (p.per_cu > 1 && (double)tiles * S <= cus) us *= kGemmAlone;
            if (S > 1) us += split.launch_us + split.mb_us * 2.0 * S * mn * 1e-6;
            if (best.mt == 0 || us < best_us) {
                best = GemmPlan{p.mt, p.nw, p.kw, S};
                best_us = us;
            }
        }
    }
    return best;
}

// Partials of a plan.
inline size_t gemm_plan_bytes(const GemmPlan &p, int M, int N) {
    return p.splits > 1 ? (size_t)(p.splits - 1) * M * N * sizeof(float) : 0;
}

}  // namespace gollek
