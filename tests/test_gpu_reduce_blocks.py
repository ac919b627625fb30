"""Box sums and residual at the edges of their block counts: fewer cells than
one block, a last block in part, every block busy, one more than that, and a
state that is read with nontemporal loads."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def reference(s, box):
    f = s.getDensityDistributions(*box).reshape(19, -1).astype(np.float64)
    cx = np.array([1, -1, 0, 0, 1, -1, 1, -1, 1, -1, 1, -1, 0, 0, 0, 0, 0, 0, 0])
    cy = np.array([0, 0, 1, -1, 1, -1, -1, 1, 0, 0, 0, 0, 1, -1, 1, -1, 0, 0, 0])
    cz = np.array([0, 0, 0, 0, 0, 0, 0, 0, 1, -1, -1, 1, 1, -1, -1, 1, 1, -1, 0])
    plane = f.sum(axis=1)
    return np.array([plane.sum(), cx @ plane, cy @ plane, cz @ plane, f.shape[1]])


@pytest.mark.parametrize("precision,size", [
    ("f32", (1, 1, 1)), ("f32", (5, 4, 3)), ("f32", (62, 14, 6)), ("f64", (126, 62, 62)),
    ("f32", (126, 62, 63)), ("f16s", (130, 70, 66)), ("f32", (154, 152, 153))])
def test_block_edges(hip, precision, size):
    print("[case] reduce blocks", precision, size, flush=True)
    s = hip.LbmSolverHIP(size, precision=precision, inv_tau=1.1, store_densities=False,
                         store_velocities=False)
    rng = np.random.default_rng(3)
    cells = size[0] * size[1] * size[2]
    w = np.array([1 / 18] * 4 + [1 / 36] * 12 + [1 / 18] * 2 + [1 / 3])
    f = w[:, None] * rng.uniform(0.97, 1.03, (19, cells)).astype(np.float32)
    s.setDensityDistributions(f.astype(s.dtype).ravel())
    full = ((0, 0, 0), s.size_h)
    for box in (full, ((1, 1, 1), size)):
        got, want = s.reduce_box(*box), reference(s, box)
        # sums of n doubles of one magnitude: n * 2^-53 relative to the mass
        assert got[4] == want[4]
        assert np.all(np.abs(got[:4] - want[:4]) <= 1e-12 * want[0])
    assert s.residual(0) == float("inf")
    before = s.getMoments(0).reshape(4, -1)[1:].astype(np.float64)
    s.setDensityDistributions((f * (1 + 1e-3 * rng.standard_normal((19, cells)))).astype(s.dtype)
                              .ravel())
    after = s.getMoments(0).reshape(4, -1)[1:].astype(np.float64)
    want = np.sqrt(((after - before) ** 2).sum() / (after ** 2).sum())
    assert abs(s.residual(0) - want) <= 1e-12 * want
    assert s.residual(0) == 0.0
    s.close()
