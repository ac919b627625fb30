// The batch autotuner's search (lbm_tuner.hpp) against made-up times: the tuning
// that is fastest by them has to be chosen. Prints what fails; returns the count.
#include <cstdio>

#include "lbm_tuner.hpp"

using namespace lbm;

static lbm_batch_tuning tuning(int block, int cells, int a, int b, int group_mb)
{
    lbm_batch_tuning t{};
    t.block = block;
    t.cells_per_thread = cells;
    t.options[0] = a;
    t.options[1] = b;
    t.group_mb = group_mb;
    return t;
}

static int failed = 0;

template <class Time>
static void expect(const char* what, const lbm_batch_tuning& start, const lbm_batch_tuning& untuned,
                   bool pairs, Time ms, const lbm_batch_tuning& want)
{
    const lbm_batch_tuning grouped = tuning(256, 2, 0, 6, 224);
    lbm_batch_tuning got{};
    int longest = 0;
    const int rc = search_tuning(
        start, untuned, grouped, 1024, 4, 3,
        [&](const lbm_batch_tuning& t, int steps, float* out) {
            longest = steps > longest ? steps : longest;
            *out = ms(t);
            return 0;
        },
        [&](const lbm_batch_tuning&) { return pairs; }, &got);
    if (rc || longest != 12 || !same_tuning(got, want)) {
        printf("%s: rc %d, %d steps, got block %d cells %d waves %d options %d %d pairs %d group %d\n",
               what, rc, longest, got.block, got.cells_per_thread, got.waves_per_cu,
               got.options[0], got.options[1], got.pairs, got.group_mb);
        failed++;
    }
}

int main()
{
    const lbm_batch_tuning untuned = tuning(256, 1, 9, 9, 0);
    const lbm_batch_tuning set = tuning(512, 2, 1, 0, 128);
    for (const lbm_batch_tuning& start : {untuned, set}) {
        // nothing beats the untuned schedule, and what it stands for is not
        // what its fields would launch by themselves
        auto untuned_best = [&](const lbm_batch_tuning& t) {
            return same_tuning(t, untuned) ? 1.0f : t.group_mb ? 1.1f : 1.4f;
        };
        expect("untuned", start, untuned, true, untuned_best, untuned);
        // only the extra candidate is fast, then a pair pass
        const lbm_batch_tuning extra = tuning(256, 2, 0, 6, 224);
        expect("extra", start, untuned, false,
               [&](const lbm_batch_tuning& t) { return same_tuning(t, extra) ? 0.9f : untuned_best(t); },
               extra);
        lbm_batch_tuning pair{};
        expect("pairs", start, untuned, true,
               [&](const lbm_batch_tuning& t) {
                   if (t.pairs == 3 && t.options[0] == 2)
                       pair = t;
                   return t.pairs == 3 && t.options[0] == 2 ? 0.8f : untuned_best(t);
               },
               pair);
        // all alike: the starting tuning
        expect("alike", start, untuned, true, [](const lbm_batch_tuning&) { return 1.0f; }, start);
    }
    // an error of a trial is the search's
    lbm_batch_tuning got{};
    int calls = 0;
    const int rc = search_tuning(
        untuned, untuned, set, 512, 4, 2,
        [&](const lbm_batch_tuning&, int, float* out) { return *out = 1.0f, ++calls == 5 ? -7 : 0; },
        [](const lbm_batch_tuning&) { return false; }, &got);
    if (rc != -7 || calls != 5) {
        printf("error of a trial: rc %d after %d calls\n", rc, calls);
        failed++;
    }
    return failed;
}
