"""Batches of 16-bit members in pairs of neighbouring cells: every workgroup
shape with an even number of cells per thread, on odd sizes with every flag,
gives each member the bits of its own plain steps."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SIZES = [(1, 1, 1), (7, 5, 3), (31, 22, 17), (64, 30, 19), (45, 44, 43)]


@pytest.mark.parametrize("block,cells,waves", [(256, 2, 0), (256, 4, 0), (512, 2, 3), (512, 4, 0),
                                               (1024, 2, 1), (256, 2, 2), (256, 1, 0)])
@pytest.mark.parametrize("outputs", [False, True])
@pytest.mark.parametrize("precision", ["f16s", "bf16s", "f16c"])
def test_pairs_of_cells_keep_the_bits(hip, precision, outputs, block, cells, waves):
    from cavityflow_cuda_amd._lib import check, lib
    from cavityflow_cuda_amd.batch import CavityBatch, CavitySpec
    print("[case] batch pairs", precision, outputs, block, cells, waves, flush=True)
    params = dict(inv_tau=1.3, velocity_dimless=(0.07, 0.0, 0.0),
                  acceleration_dimless=(1e-4, 0.0, -2e-4))
    b = CavityBatch([CavitySpec(z, 0.07, 150.0, params) for z in SIZES], precision,
                    store_outputs=outputs)
    b.set_tuning(block=block, cells_per_thread=cells, waves_per_cu=waves, options=(1, 2))
    rng = np.random.default_rng(3)
    w = np.array([1 / 18] * 4 + [1 / 36] * 12 + [1 / 18] * 2 + [1 / 3], np.float32)
    alone = []
    for size, s in zip(SIZES, b.solvers):
        n = int(np.prod([v + 2 for v in size]))
        flags = rng.choice(np.array([1, 2, 4, 8], np.int32), n, p=[0.2, 0.65, 0.1, 0.05])
        dd = (w[:, None] * rng.uniform(0.95, 1.05, n).astype(np.float32)[None, :]).ravel()
        p = hip.LbmSolverHIP(size, precision=precision, inv_tau=1.3, lid_velocity=0.07,
                             gravitation=params["acceleration_dimless"],
                             store_densities=outputs, store_velocities=outputs)
        for k in (0, 1):
            check(lib().lbm_set_launch_options(p.handle, k, 0))
        for x in (s, p):
            x.setFlags(flags, (0, 0, 0), x.size_h)
            x.setDensityDistributions(dd, (0, 0, 0), x.size_h)
        alone.append(p)
    b.run(4)
    for p in alone:
        for step in range(4):
            (p.simulationStepBeta if step & 1 else p.simulationStepAlpha)()
    for s, p in zip(b.solvers, alone):
        assert np.array_equal(s.save_state(), p.save_state())
        if outputs:
            assert np.array_equal(s.getVelocities(), p.getVelocities())
            assert np.array_equal(s.getDensities(), p.getDensities())
        p.close()
    b.close()
