"""Batches without a set tuning: several groups, one of them a member larger
than the last-level cache, give every member the bits of one plain launch over
all members; single half-steps too."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SIZES = {"f32": [(101, 99, 97), (40, 33, 21), (153, 150, 149), (97, 88, 90), (1, 1, 1)],
         "f64": [(84, 81, 80), (90, 70, 60), (17, 5, 9)],
         "f16s": [(130, 120, 125), (130, 110, 120), (64, 64, 64), (140, 150, 130)],
         "f16c": [(130, 120, 125), (37, 20, 11), (150, 140, 130)]}


@pytest.mark.parametrize("precision", sorted(SIZES))
def test_untuned_groups_match_one_plain_launch(hip, precision):
    from cavityflow_cuda_amd._lib import check, lib
    from cavityflow_cuda_amd.batch import CavityBatch, CavitySpec
    print("[case] batch groups", precision, flush=True)
    states = []
    for tuned in (False, True):
        params = dict(inv_tau=1.3, velocity_dimless=(0.07, 0.0, 0.0),
                      acceleration_dimless=(0.0, 0.0, 0.0))
        specs = [CavitySpec(z, 0.07, 150.0, params) for z in SIZES[precision]]
        b = CavityBatch(specs, precision)
        if tuned:
            b.set_tuning(options=(0, 0))
        b.run(6)
        for phase in (0, 1):
            check(lib().lbm_batch_step(b._h, phase, None))
        b.run(2)
        states.append([s.save_state() for s in b.solvers])
        b.close()
    for i, (a, c) in enumerate(zip(*states)):
        assert np.array_equal(a, c), i
