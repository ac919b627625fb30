// The batch autotuner's search (lbm_batch.hip): host code that sees the GPU only
// through the times it asks for.
#pragma once

#include <algorithm>
#include <limits>
#include <utility>
#include <vector>

#include "lbm_abi.h"

namespace lbm {

inline bool same_tuning(const lbm_batch_tuning& a, const lbm_batch_tuning& b)
{
    return a.block == b.block && a.cells_per_thread == b.cells_per_thread &&
           a.waves_per_cu == b.waves_per_cu && a.options[0] == b.options[0] &&
           a.options[1] == b.options[1] && a.pairs == b.pairs && a.group_mb == b.group_mb;
}

// candidates besides the starting tuning and the untuned schedule that the final
// round times again over longer runs
constexpr size_t kFinalists = 4;

// Trials time whole steps (alpha then beta), since each phase's speed depends on
// what the other leaves in the caches: first the workgroup shape with the launch
// options of `start`, then alpha's options with beta's fixed, then beta's with the
// chosen alpha, then member groups and the shapes again under the chosen group,
// then the pair pass. `untuned` stands for the schedule of a batch without a set
// tuning: it chooses options for each group and may run beta's tiles backwards,
// which no other tuning says, so it is timed as it is, never varied, and always
// one of the finalists. `grouped` is one more candidate.
//   time(tuning, steps, &ms): ms per whole step, an LBM_* code
//   allowed(tuning): whether the members allow its pair pass
template <class Time, class Allowed>
int search_tuning(const lbm_batch_tuning& start, const lbm_batch_tuning& untuned,
                  const lbm_batch_tuning& grouped, int max_block, int pair_shapes,
                  int trial_steps, Time time, Allowed allowed, lbm_batch_tuning* chosen)
{
    int rc;
    lbm_batch_tuning best = start;
    float best_step = std::numeric_limits<float>::infinity();
    std::vector<std::pair<float, lbm_batch_tuning>> timed;   // every trial, for the final round
    auto consider = [&](const lbm_batch_tuning& c) -> int {
        if (same_tuning(c, untuned))
            return LBM_OK;   // a finalist
        float t = 0.f;
        const int r = time(c, trial_steps, &t);
        if (r)
            return r;
        timed.push_back({t, c});
        if (t < best_step) {
            best_step = t;
            best = c;
        }
        return LBM_OK;
    };
    // at most two 1024-thread workgroups are resident per CU
    for (int blk : {256, 512, 1024})
        for (int cpt : {1, 2, 4})
            for (int wpc : {0, 1, 2, 3, 4, 8, 16}) {
                if (blk > max_block || (blk == 1024 && wpc > 2))
                    continue;
                lbm_batch_tuning cand = start;
                cand.block = blk;
                cand.cells_per_thread = cpt;
                cand.waves_per_cu = wpc;
                if ((rc = consider(cand)))
                    return rc;
            }
    for (int ph = 0; ph < 2; ph++) {
        const lbm_batch_tuning shape = best;
        for (int opt : {0, 1, 2, 3, 4, 5, 6, 8, 9, 16, 17}) {
            lbm_batch_tuning cand = shape;
            cand.options[ph] = opt;
            if ((rc = consider(cand)))
                return rc;
        }
    }
    // member groups small enough for the last-level cache to keep their state
    // between consecutive steps
    const lbm_batch_tuning ungrouped = best;
    for (int mb : {32, 64, 128, 192, 256, 384}) {
        lbm_batch_tuning cand = ungrouped;
        cand.group_mb = mb;
        if ((rc = consider(cand)))
            return rc;
    }
    if ((rc = consider(grouped)))
        return rc;
    // with the state of a group in the cache the best workgroup shape can
    // differ from the streaming one: the shapes once more, grouped
    if (best.group_mb > 0) {
        const lbm_batch_tuning shape = best;
        for (int blk : {256, 512, 1024})
            for (int cpt : {1, 2, 4}) {
                if (blk > max_block || (blk == 1024 && shape.waves_per_cu > 2))
                    continue;
                lbm_batch_tuning cand = shape;
                cand.block = blk;
                cand.cells_per_thread = cpt;
                if ((rc = consider(cand)))
                    return rc;
            }
    }
    // the pair pass, when the members allow it (else: the in-place launches)
    bool eligible = true;
    for (int shape = 1; shape <= pair_shapes && eligible; shape++)
        for (int opt = 0; opt < 4 && eligible; opt++) {
            lbm_batch_tuning cand = best;
            cand.pairs = shape;
            cand.group_mb = 0;
            cand.options[0] = opt;
            eligible = allowed(cand);
            if (eligible && (rc = consider(cand)))
                return rc;
        }
    // Short trials are noisy, and the more candidates, the likelier a lucky
    // trial wins: the few fastest distinct candidates, the starting tuning and
    // the untuned schedule run again over longer runs, interleaved, and the
    // least total time wins (the starting tuning on a tie).
    std::stable_sort(timed.begin(), timed.end(),
                     [](const auto& x, const auto& y) { return x.first < y.first; });
    std::vector<lbm_batch_tuning> finalists{start};
    if (!same_tuning(start, untuned))
        finalists.push_back(untuned);
    const size_t most = finalists.size() + kFinalists;
    for (const auto& tc : timed) {
        if (finalists.size() == most)
            break;
        bool seen = false;
        for (const lbm_batch_tuning& f : finalists)
            seen = seen || same_tuning(f, tc.second);
        if (!seen)
            finalists.push_back(tc.second);
    }
    const int long_steps = 4 * trial_steps;
    std::vector<float> total(finalists.size(), 0.f);
    for (int rep = 0; rep < 2; rep++)
        for (size_t i = 0; i < finalists.size(); i++) {
            float t = 0.f;
            if ((rc = time(finalists[i], long_steps, &t)))
                return rc;
            total[i] += t;
        }
    size_t win = 0;
    for (size_t i = 1; i < finalists.size(); i++)
        if (total[i] < total[win])
            win = i;
    *chosen = finalists[win];
    return LBM_OK;
}

}  // namespace lbm
