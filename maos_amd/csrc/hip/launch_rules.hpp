// Rules that choose the launch shape of a batch.  None of these choices
// changes a result.  Host code without HIP.
#pragma once
#include <algorithm>
#include <utility>
#include <vector>

namespace mtk {

constexpr int TILE = 16;      // output tile edge of the WFS / layer passes
constexpr int LTY = 64;       // tile height of the 16 x 64 layer kernel (k_layer_m8)
constexpr int LTY2 = 32;      // tile height of the 16 x 32 layer kernel (k_layer_m8)

// One job of a batch, as the layer pass sees it.
struct LayerJob {
    bool matched;       // matched rays; others take the generic kernel (TILE)
    int tuned;          // chosen tile rows, 0: by the rule
    bool fits2, fits;   // LTY2-row, LTY-row tiles fit every layer
    long nodes;         // layer nodes of its systems
};

// Layer tile rows of each job.  Without a tuned choice: TILE rows, in the
// split form where that applies, for a few small systems, LTY2 from about
// 100 000 nodes in the launch on, whether they are one plan's systems or many
// plans' (the kernel sees workgroups).  k_layer, us, 16 / 32 rows (64): 5184 nodes a
// system, 1 system 4.8 5.4, 16: 5.7 6.3, 32: 7.0 6.2, 256: 25.9 15.1; 6272
// nodes, 16: 6.2 5.6; 16 384 nodes, 1: 5.1 5.6, 8: 6.1 5.6, 64: 19.7 11.3; the
// 30 m system, 1: 5.7 6.1 (12.4), 8: 11.4 8.5 (12.4), 32: 31.3 17.5 (19.3), 256:
// 201 88 (91).  Jobs that stay on TILE rows (layers under LTY2 + 2 rows, a tuned
// choice) are then a launch of their own, which has to be repaid: a group of
// 8 small members (28-row layers) and 4 / 8 / 16 / 24 of 30 m, 10 iterations,
// all on 16 rows against large ones on 32: 713 841 1051 1307 against 750 867 1020
// 1248 us; 16 / 32 of 20 m: 647 889 against 688 892.
constexpr long LTY2_NODES = 100000, LTY2_NODES_BESIDE = 600000;
inline std::vector<int> layer_rows(const std::vector<LayerJob> &jobs) {
    auto stays = [](const LayerJob &j) { return j.tuned == TILE || (!j.fits2 && j.tuned != LTY); };
    long nodes = 0;      // of the LTY2 launch
    bool beside = false;  // a TILE launch whatever the others do
    for (const LayerJob &j : jobs) {
        if (!j.matched) continue;
        if (stays(j)) beside = true;
        else if (j.tuned != LTY) nodes += j.nodes;
    }
    const int built_in = nodes >= (beside ? LTY2_NODES_BESIDE : LTY2_NODES) ? LTY2 : TILE;
    std::vector<int> rows;
    for (const LayerJob &j : jobs) {
        if (!j.matched || stays(j)) rows.push_back(TILE);
        else if (j.tuned == LTY) rows.push_back(j.fits ? LTY : TILE);
        else rows.push_back(j.tuned ? j.tuned : built_in);
    }
    return rows;
}

inline int ceil_div(int a, int b) { return (a + b - 1) / b; }

// Systems per workgroup: the most of cmax, cmax/2, .., 1 that keeps >= thresh
// workgroups in the launch (thresh4 for 4 systems) and leaves at most a fifth
// of their slots empty; jw = (workgroups per system, systems) per job.  The
// kernels compute an empty slot like a filled one and drop it: groups of 8 / 16
// / 32 one-system 30 m members, 10 iterations, with 2, 2, 4 slots (as the number
// of workgroups alone would have it) 471 718 1143 us, with one 450 583 915.
inline int pick_cs(const std::vector<std::pair<long, int>> &jw, int cmax, int thresh, int thresh4) {
    for (int cs = cmax; cs > 1; cs >>= 1) {
        long tot = 0, filled = 0;
        for (auto &p : jw) {
            tot += p.first * ceil_div(p.second, cs);
            filled += p.first * p.second;
        }
        if (tot >= (cs == 4 ? thresh4 : thresh) && 5 * filled >= 4 * cs * tot) return cs;
    }
    return 1;
}

// The group autotuner's search: coordinate descent from the built-in choice
// over the column kernel, the layer tile rows, then the systems per workgroup
// of the WFS and layer passes; a change is kept when it saves more than 2 %.
// timed: the time of a choice, in gpu_tomo_tune_set's order.  A tile shape that
// fits no member (fits2, fits: LTY2, LTY rows fit one) would be TILE rows again.
template <typename Timed> void group_descent(bool fits2, bool fits, Timed timed, int *best) {
    const int start[6] = {0, 0, 0, 0, 0, 1};
    std::copy(start, start + 6, best);
    double tbest = timed((const int *)best);
    auto trial = [&](int k, const std::vector<int> &vals) {
        for (int v : vals) {
            if (v == best[k]) continue;
            int c[6];
            std::copy(best, best + 6, c);
            c[k] = v;
            const double t = timed((const int *)c);
            if (t < tbest * 0.98) {
                tbest = t;
                best[k] = v;
            }
        }
    };
    trial(4, {2});
    std::vector<int> rows;
    if (fits) rows.push_back(LTY);
    if (fits2) rows.push_back(LTY2);
    rows.push_back(TILE);
    trial(3, rows);
    trial(0, {1, 2, 4});
    trial(1, {1, 2, 4});
}

}  // namespace mtk
