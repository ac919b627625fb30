"""Alpha and beta where the collision branches on a whole wave: lid cells and
non-finite densities among ordinary ones, with and without gravity, against
the oracle (NaN and infinities in the same places, every other value's bits)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

PREC = {np.float32: "f32", np.float64: "f64"}


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("gravity", [(0.0, 0.0, 0.0), (0.0, -0.0, 0.0), (0.0, 0.0, 3e-4)])
@pytest.mark.parametrize("size", [(62, 3, 4), (13, 6, 5)])
def test_lid_and_non_finite_cells_match_oracle(hip, oracle_cpu, dtype, gravity, size):
    print("[case] edges", dtype.__name__, gravity, size, flush=True)
    rng = np.random.default_rng(17)
    kw = dict(inv_tau=1.21, lid_velocity=0.05, gravitation=gravity)
    o = oracle_cpu.OracleSolver(size, (1,) * 6, dtype=dtype, **kw)
    o.dd[:] = (rng.random(o.dd.size) * 0.08 + 0.01).astype(dtype)
    o.flags[:] = rng.choice([1, 2, 2, 2, 4, 8], size=o.n).astype(np.int32)
    for value in (np.inf, -np.inf, np.nan):
        o.dd[rng.integers(0, o.dd.size, 2)] = value
    s = hip.LbmSolverHIP(size, (1,) * 6, PREC[dtype], kw["inv_tau"], kw["lid_velocity"], gravity)
    box = ((0, 0, 0), s.size_h)
    s.setDensityDistributions(o.dd, *box)
    s.setFlags(o.flags, *box)
    s.setVelocities(o.u, *box)
    s.setDensities(o.rho, *box)
    with np.errstate(all="ignore"):
        for step in range(4):
            if step & 1:
                o.beta()
                s.simulationStepBeta()
            else:
                o.alpha()
                s.simulationStepAlpha()
            for got, want in ((s.getDensityDistributions(*box), o.dd),
                              (s.getVelocities(*box), o.u), (s.getDensities(*box), o.rho)):
                nan = np.isnan(want)
                assert np.array_equal(np.isnan(got), nan), step
                got, want = np.where(nan, 0, got), np.where(nan, 0, want)
                assert got.tobytes() == want.tobytes(), step
    s.close()
