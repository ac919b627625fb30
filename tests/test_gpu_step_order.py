"""Beta from the last cells to the first, and the XCD map of both steps of small
domains: whatever shape the sizes and the steps in between choose gives the bits
of plain launches."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# one size for each line of the choice: within the L2s (with and without the
# map), larger than the Infinity Cache up to the sizes that stream
SIZES = [("f32", (24, 90, 89), False), ("f32", (62, 62, 62), True), ("f64", (51, 49, 50), False),
         ("f16s", (75, 74, 73), True), ("f16c", (91, 87, 83), False),
         ("f32", (151, 149, 150), False), ("f32", (229, 186, 141), True),
         ("f32", (247, 250, 239), False), ("f32", (281, 280, 279), False),
         ("f64", (151, 150, 139), True), ("f64", (181, 180, 179), False),
         ("f64", (233, 232, 231), False), ("f16s", (205, 203, 199), True),
         ("bf16s", (241, 260, 277), True), ("f16s", (321, 319, 320), False),
         ("f16c", (321, 319, 320), False), ("f16c", (221, 219, 220), False)]


@pytest.fixture(scope="module")
def neighbour(hip):
    """A solver of 348 MB: one half-step of it empties the Infinity Cache."""
    s = hip.LbmSolverHIP((164, 164, 164), store_densities=False, store_velocities=False)
    yield s
    s.close()


def solver(hip, precision, size, outputs):
    s = hip.LbmSolverHIP(size, precision=precision, inv_tau=1.3, lid_velocity=0.07,
                         store_densities=outputs, store_velocities=outputs)
    s.setDrivenCavitySzenario()
    w = np.array([1 / 18] * 4 + [1 / 36] * 12 + [1 / 18] * 2 + [1 / 3], s.dtype)
    noise = np.random.default_rng(5).random(size[0] * size[1] * size[2], np.float32)
    s.setDensityDistributions((w[:, None] * (noise * 0.04 + 0.98)[None, :].astype(s.dtype)).ravel())
    return s


@pytest.mark.parametrize("visits", [False, True])
@pytest.mark.parametrize("precision,size,outputs", SIZES)
def test_order_of_cells_keeps_the_bits(hip, neighbour, precision, size, outputs, visits):
    from cavityflow_cuda_amd._lib import check, lib
    print("[case] step order", precision, size, outputs, visits, flush=True)
    chosen, plain = (solver(hip, precision, size, outputs) for _ in range(2))
    for k in (0, 1):
        check(lib().lbm_set_launch_options(plain.handle, k, 0))
    for s in (chosen, plain):
        for step in range(4):
            if visits and step % 2 == 0:
                neighbour.simulationStepAlpha()
            (s.simulationStepBeta if step & 1 else s.simulationStepAlpha)()
    assert np.array_equal(chosen.save_state(), plain.save_state())
    if outputs:
        assert np.array_equal(chosen.getVelocities(), plain.getVelocities())
        assert np.array_equal(chosen.getDensities(), plain.getDensities())
    chosen.close()
    plain.close()


@pytest.mark.parametrize("precision", ["f32", "f64", "f16s"])
@pytest.mark.parametrize("split", [(2, 1, 1), (1, 3, 1), (2, 2, 2)])
def test_split_cavity_matches_the_undivided_one(hip, precision, split):
    """Subdomains stepped forwards by alpha and backwards by beta, together
    larger than the Infinity Cache (FP32 and FP64)."""
    from cavityflow_cuda_amd.controller import CavityController
    print("[case] split order", precision, split, flush=True)
    size = (168, 162, 166)
    fields = []
    for parts in ((1, 1, 1), split):
        c = CavityController(size, 0.05, 300.0, precision, split=parts)
        for _ in range(6):
            c.computeNextStep()
        c.sync()
        fields.append((c.getVelocities(), c.getDensities()))
        c.close()
    assert np.array_equal(fields[0][0], fields[1][0])
    assert np.array_equal(fields[0][1], fields[1][1])
