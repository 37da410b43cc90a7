// The matmul planner: launch shape and K split of the tiled / ring kernels
// (k_gemm.hip) from estimated launch times. Host code only.
#pragma once
#include <cstddef>
#include <cstdint>

namespace spq4k {

constexpr int REDUCE_MAX_SPLIT = 32;   // K ranges the reduction pass sums

// What a launch shape costs (us), for plan_shape's estimate: `t0`, fill and
// drain of a round; `t1`, a super-block's step with one workgroup a CU; `tn`, with
// `occ` workgroups a CU (as many as its LDS leaves room for). rows and tok: the
// workgroup's tile, powers of two. The K-quants' are fitted together with their
// PlanCosts to the times of 17,500 launches on an MI355X (256 CUs, cold weights;
// 1609 matmuls of 128..60000 rows, 1..54 super-blocks, 4..5000 tokens, each with up
// to four K splits of every shape near the best) so that the least estimate is
// the least time: its choice is 0.4 / 0.3 / 0.1% slower than the fastest of those
// launches on average (Q4_K / Q5_K / Q6_K), more than 4% for 31 matmuls and at
// most 10%. Steps timed one shape at a time with 4 us a round, which these
// replace, chose 3.1 / 2.3 / 2.8% slower ones, more than 4% for 471 and up to 24%.
// Shapes that no size prefers are not listed.
struct ShapeCost {
    int cfg, rows, tok, occ;
    float t0, t1, tn;
};
constexpr ShapeCost kCostQ4K[] = {{8, 64, 16, 3, 0.4f, 0.53f, 1.35f}, {6, 128, 16, 2, 0.8f, 0.75f, 1.66f},
                                  {37, 64, 32, 4, 0.5f, 0.68f, 1.72f}, {33, 64, 64, 2, 1.6f, 1.16f, 1.49f},
                                  {32, 128, 64, 2, 2.8f, 1.61f, 2.50f}, {1, 128, 64, 1, 1.5f, 1.70f, 1.70f}};
constexpr ShapeCost kCostQ6K[] = {{29, 64, 16, 2, 1.8f, 0.85f, 1.58f}, {16, 128, 32, 1, 3.4f, 1.71f, 1.71f},
                                  {38, 64, 32, 2, 1.5f, 1.25f, 1.91f}, {34, 64, 64, 2, 3.4f, 1.40f, 1.90f},
                                  {17, 256, 64, 1, 4.7f, 4.66f, 4.66f}};
constexpr ShapeCost kCostQ5K[] = {{30, 64, 16, 2, 1.2f, 0.78f, 1.36f}, {20, 128, 16, 1, 1.8f, 1.25f, 1.25f},
                                  {39, 64, 32, 3, 1.4f, 0.96f, 2.29f}, {35, 64, 64, 2, 2.1f, 1.49f, 2.45f}};
// Q8_0: steps timed one shape at a time, 4 us a round. The fit would choose 1.1%
// faster launches on average (4096 x 4096 at T = 40 16.2 us against 18.9), but with
// fewer K ranges, whose longer serial sums of 32-value blocks are further from the
// 64-bit result there (1.1e-7 against 9.5e-8).
constexpr ShapeCost kCostQ80[] = {{31, 64, 16, 2, 4.0f, 1.40f, 1.74f}, {28, 128, 16, 2, 4.0f, 2.21f, 3.24f},
                                  {40, 64, 32, 2, 4.0f, 1.83f, 2.01f}, {36, 64, 64, 2, 4.0f, 3.31f, 3.54f}};

// The costs of a weight format: its shapes, each further workgroup a CU starts in
// a round (us), the reduction launch of a K split (us) and the bytes it reads
// and writes in a us.
struct PlanCosts {
    const ShapeCost* shape;
    int n;
    float place_us, reduce_us, reduce_bytes;
};
template <int N>
constexpr PlanCosts plan_costs(const ShapeCost (&shape)[N], float place_us, float reduce_us, float reduce_bytes) {
    return {shape, N, place_us, reduce_us, reduce_bytes};
}
constexpr PlanCosts kPlanQ4K = plan_costs(kCostQ4K, 0.4f, 2.5f, 2.2e6f);
constexpr PlanCosts kPlanQ5K = plan_costs(kCostQ5K, 0.4f, 2.5f, 2.2e6f);
constexpr PlanCosts kPlanQ6K = plan_costs(kCostQ6K, 0.4f, 2.5f, 2.2e6f);
constexpr PlanCosts kPlanQ80 = plan_costs(kCostQ80, 0.0f, 3.0f, 3.5e6f);

struct ShapePlan {
    int cfg, ksplit, kchunk;   // kchunk super-blocks a K range
};

// The shape and K split of least estimated time for n matrices of M[i] rows
// and nb super-blocks a row, T tokens. A launch runs in rounds of occ
// workgroups a CU: a round costs its fill and drain, the further workgroups a CU
// starts, and a step a super-block, the last round less when it leaves CUs (or
// their second place) empty; a K split adds the reduction pass. So a grid a
// little over a whole number of rounds takes fewer ranges or another tile.
//
// This runs on the host in every matmul call, so the splits and their reduction
// are worked out once for all shapes, and a split whose bound (one round of
// `t1` steps) already costs more than the best is not priced: a Q4_K plan of
// 24576 x 4096 at T = 5 takes 0.31 us, of 6144 x 4096 0.24, a Q6_K one of 4096 x
// 12288 at T = 100 0.16 (2.7 GHz Xeon); all shapes and splits priced one by one,
// two divisions each, took 0.82, 0.84 and 0.33.
inline ShapePlan plan_shape(const PlanCosts& p, int n, const int32_t* M, int nb, int64_t T, int num_cus,
                            size_t max_partial_bytes) {
    size_t rows = 0;
    for (int i = 0; i < n; ++i) rows += (size_t)M[i];
    const size_t per_split = (size_t)T * rows * sizeof(float);
    const size_t fit = max_partial_bytes / per_split;
    const int most = fit < 1 ? 1 : fit < REDUCE_MAX_SPLIT ? (int)fit : REDUCE_MAX_SPLIT;
    int ks[REDUCE_MAX_SPLIT], chunk[REDUCE_MAX_SPLIT], splits = 0;
    float reduce[REDUCE_MAX_SPLIT];
    for (unsigned want = 1; want <= (unsigned)most && want <= (unsigned)nb; ++want) {
        const unsigned kc = ((unsigned)nb + want - 1) / want;
        if (((unsigned)nb + kc - 1) / kc != want) continue;   // the same ranges as a smaller count
        ks[splits] = (int)want;
        chunk[splits] = (int)kc;
        reduce[splits] = want > 1 ? p.reduce_us + (float)(want + 1) * (float)per_split / p.reduce_bytes : 0.0f;
        ++splits;
    }
    ShapePlan g = {-1, 1, nb};
    float best = 0.0f;
    for (int k = 0; k < p.n; ++k) {
        const ShapeCost& c = p.shape[k];
        int64_t tiles = 0;
        for (int i = 0; i < n; ++i) tiles += ((int64_t)M[i] + c.rows - 1) / (unsigned)c.rows;
        tiles *= (T + c.tok - 1) / (unsigned)c.tok;
        const unsigned place = (unsigned)num_cus * (unsigned)c.occ;
        const int64_t full1 = tiles / place;
        const unsigned rem1 = (unsigned)(tiles - full1 * place);
        for (int s = 0; s < splits; ++s) {
            if (g.cfg >= 0 && c.t0 + c.t1 * (float)chunk[s] + reduce[s] >= best) {
                if (c.t0 + reduce[s] >= best) break;
                continue;
            }
            const unsigned over = rem1 * (unsigned)ks[s], more = over / place, rem = over - more * place;
            const int64_t full = full1 * ks[s] + more;
            float step = (float)full * c.tn;
            int on = 0;
            if (rem > 0) {   // the fullest CU of the last round sets its pace
                on = 1;
                while (rem > (unsigned)(on * num_cus)) ++on;
                step += on == 1 ? c.t1 : c.t1 + (c.tn - c.t1) * (float)(on - 1) / (float)(c.occ - 1);
            }
            const float us = c.t0 * (float)(full + (on > 0)) +
                             p.place_us * (float)(full * (c.occ - 1) + (on > 1 ? on - 1 : 0)) + step * (float)chunk[s] +
                             reduce[s];
            if (g.cfg < 0 || us < best) {
                best = us;
                g = {c.cfg, ks[s], ks[s] > 1 ? chunk[s] : nb};
            }
        }
    }
    return g;
}

}  // namespace spq4k
