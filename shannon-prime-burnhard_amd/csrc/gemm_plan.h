// The matmul planner: launch shape and K split of the tiled / ring kernels
// (k_gemm.hip) from estimated launch times. Host code only.
#pragma once
#include <cstddef>
#include <cstdint>

namespace spq4k {

constexpr int REDUCE_MAX_SPLIT = 32;   // K ranges the reduction pass sums

// What a launch shape costs, measured on an MI355X (256 CUs, cold weights, one
// K range, 8 and 24 super-blocks a row; us): `t1`, a super-block's step of a
// launch with one workgroup a CU; `tn`, of one with `occ` workgroups a CU (as
// many as its LDS leaves room for). rows and tok: the workgroup's tile, powers
// of two.
struct ShapeCost {
    int cfg, rows, tok, occ;
    float t1, tn;
};
constexpr ShapeCost kCostQ4K[] = {{8, 64, 16, 3, 0.60f, 1.45f},  {6, 128, 16, 2, 0.90f, 1.86f},
                                  {7, 128, 32, 1, 1.15f, 1.15f}, {1, 128, 64, 1, 1.70f, 1.70f},
                                  {32, 128, 64, 2, 1.76f, 3.14f}, {11, 256, 64, 1, 3.13f, 3.13f},
                                  {37, 64, 32, 4, 0.80f, 2.54f}, {33, 64, 64, 2, 1.08f, 1.76f}};
constexpr ShapeCost kCostQ6K[] = {{29, 64, 16, 2, 0.92f, 1.57f}, {18, 64, 64, 1, 1.65f, 1.65f},
                                  {16, 128, 32, 1, 1.79f, 1.79f}, {14, 128, 64, 1, 2.20f, 2.20f},
                                  {17, 256, 64, 1, 4.66f, 4.66f}, {38, 64, 32, 2, 1.15f, 1.92f},
                                  {34, 64, 64, 2, 1.57f, 2.27f}};
constexpr ShapeCost kCostQ5K[] = {{30, 64, 16, 2, 0.80f, 1.28f}, {20, 128, 16, 1, 1.21f, 1.21f},
                                  {23, 64, 64, 1, 1.34f, 1.34f}, {21, 128, 32, 1, 1.60f, 1.60f},
                                  {19, 128, 64, 1, 2.19f, 2.19f}, {39, 64, 32, 3, 0.94f, 2.25f},
                                  {35, 64, 64, 2, 1.37f, 2.33f}};
constexpr ShapeCost kCostQ80[] = {{31, 64, 16, 2, 1.40f, 1.74f}, {28, 128, 16, 2, 2.21f, 3.24f},
                                  {27, 64, 64, 1, 3.37f, 3.37f}, {26, 128, 64, 1, 4.23f, 4.23f},
                                  {40, 64, 32, 2, 1.83f, 2.01f}, {36, 64, 64, 2, 3.31f, 3.54f}};

struct ShapePlan {
    int cfg, ksplit, kchunk;   // kchunk super-blocks a K range
};

// The shape and K split of least estimated time for n matrices of M[i] rows
// and nb super-blocks a row, T tokens. A launch runs in rounds of occ
// workgroups a CU; a round costs its fill and drain (4 us: the 512-tile runs of
// the sweep above against the 256-tile ones) and a step a super-block, the last
// round less when it leaves CUs (or their second place) empty; a K split adds
// the reduction pass (3 us and its bytes at 3.5 TB/s). So a grid a little over a
// whole number of rounds takes fewer ranges or another tile instead: 4096 x
// 12288 Q6_K at T = 100 ran 320 workgroups, one a CU, in two rounds of ten
// super-blocks; four ranges make one of twelve.
//
// This runs on the host in every matmul call, so the splits and their reduction
// are worked out once for all shapes, and a split whose bound (one round of
// `t1` steps) already costs more than the best is not priced: a Q4_K plan of
// 24576 x 4096 at T = 5 takes 0.37 us against 0.82, of 6144 x 4096 0.26 against
// 0.84, a Q6_K one of 4096 x 12288 at T = 100 0.20 against 0.33 (2.7 GHz Xeon).
inline ShapePlan plan_shape(const ShapeCost* cost, int ncost, int n, const int32_t* M, int nb, int64_t T, int num_cus,
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
        reduce[splits] = want > 1 ? 3.0f + (float)(want + 1) * (float)per_split / 3.5e6f : 0.0f;
        ++splits;
    }
    ShapePlan g = {-1, 1, nb};
    float best = 0.0f;
    for (int k = 0; k < ncost; ++k) {
        const ShapeCost& c = cost[k];
        int64_t tiles = 0;
        for (int i = 0; i < n; ++i) tiles += ((int64_t)M[i] + c.rows - 1) / (unsigned)c.rows;
        tiles *= (T + c.tok - 1) / (unsigned)c.tok;
        const unsigned place = (unsigned)num_cus * (unsigned)c.occ;
        const int64_t full1 = tiles / place;
        const unsigned rem1 = (unsigned)(tiles - full1 * place);
        for (int s = 0; s < splits; ++s) {
            if (g.cfg >= 0 && 4.0f + c.t1 * (float)chunk[s] + reduce[s] >= best) {
                if (4.0f + reduce[s] >= best) break;
                continue;
            }
            const unsigned over = rem1 * (unsigned)ks[s], more = over / place, rem = over - more * place;
            const int64_t full = full1 * ks[s] + more;
            float step = (float)full * c.tn;
            if (rem > 0) {   // the fullest CU of the last round sets its pace
                int on = 1;
                while (rem > (unsigned)(on * num_cus)) ++on;
                step += on == 1 ? c.t1 : c.t1 + (c.tn - c.t1) * (float)(on - 1) / (float)(c.occ - 1);
            }
            const float us = 4.0f * (float)(full + (rem > 0)) + step * (float)chunk[s] + reduce[s];
            if (g.cfg < 0 || us < best) {
                best = us;
                g = {c.cfg, ks[s], ks[s] > 1 ? chunk[s] : nb};
            }
        }
    }
    return g;
}

}  // namespace spq4k
