"""Whole-domain steps choose their launch shape from the bytes stepped between
two half-steps of a solver. Each choice gives the bits of plain launches."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# (precision, interior size): up to the L2s; within the Infinity Cache; beyond
# it (the second FP64 size is the one between both)
SIZES = [("f32", (37, 20, 11)), ("f32", (86, 83, 81)), ("f32", (163, 157, 150)),
         ("f64", (70, 69, 67)), ("f64", (121, 123, 119)), ("f64", (150, 147, 139)),
         ("f16s", (107, 103, 101)), ("f16s", (190, 187, 193)), ("f16c", (107, 103, 101)),
         ("f16c", (190, 187, 193)), ("bf16s", (107, 103, 101))]


@pytest.fixture(scope="module")
def neighbour(hip):
    """A solver of 348 MB: one half-step of it empties the Infinity Cache."""
    s = hip.LbmSolverHIP((164, 164, 164), store_densities=False, store_velocities=False)
    yield s
    s.close()


def solver(hip, precision, size, seed):
    s = hip.LbmSolverHIP(size, precision=precision, inv_tau=1.3, lid_velocity=0.07,
                         store_densities=False, store_velocities=False)
    s.setDrivenCavitySzenario()
    w = np.array([1 / 18] * 4 + [1 / 36] * 12 + [1 / 18] * 2 + [1 / 3])
    cells = size[0] * size[1] * size[2]
    noise = np.random.default_rng(seed).uniform(0.98, 1.02, cells)
    s.setDensityDistributions((w[:, None] * noise[None, :]).astype(s.dtype).ravel())
    return s


@pytest.mark.parametrize("turns", ["alone", "visits", "round_robin"])
@pytest.mark.parametrize("precision,size", SIZES)
def test_chosen_options_give_the_plain_bits(hip, neighbour, precision, size, turns):
    from cavityflow_cuda_amd._lib import check, lib
    chosen, plain = (solver(hip, precision, size, 5) for _ in range(2))
    for k in (0, 1):
        check(lib().lbm_set_launch_options(plain.handle, k, 0))
    for step in range(6):
        if turns == "round_robin" or (turns == "visits" and step % 2 == 0):
            neighbour.simulationStepAlpha()
        for s in (chosen, plain) if turns == "round_robin" else (chosen,):
            (s.simulationStepBeta if step & 1 else s.simulationStepAlpha)()
    if turns != "round_robin":   # the reference run must not come between
        for step in range(6):
            (plain.simulationStepBeta if step & 1 else plain.simulationStepAlpha)()
    a, b = chosen.save_state(), plain.save_state()
    chosen.close()
    plain.close()
    assert np.array_equal(a, b)


@pytest.mark.parametrize("turns", ["alone", "visits", "round_robin"])
@pytest.mark.parametrize("gravity", [(0.0, 0.0, 0.0), (1e-4, -2e-4, 5e-5)])
@pytest.mark.parametrize("outputs", [False, True])
@pytest.mark.parametrize("precision", ["f16s", "bf16s", "f16c"])
def test_two_cells_per_thread_with_every_flag(hip, neighbour, precision, outputs, gravity, turns):
    """The 16-bit steps' pairs of cells where one cell of a pair stores and the
    other does not, on an odd number of cells."""
    from cavityflow_cuda_amd._lib import check, lib
    size = (107, 103, 101)
    rng = np.random.default_rng(8)
    n = int(np.prod([v + 2 for v in size]))
    flags = rng.choice(np.array([1, 2, 4, 8], np.int32), n, p=[0.2, 0.65, 0.1, 0.05])
    w = np.array([1 / 18] * 4 + [1 / 36] * 12 + [1 / 18] * 2 + [1 / 3], np.float32)
    dd = (w[:, None] * rng.uniform(0.95, 1.05, n).astype(np.float32)[None, :]).ravel()
    pair = []
    for _ in range(2):
        s = hip.LbmSolverHIP(size, precision=precision, inv_tau=1.37, lid_velocity=0.04,
                             gravitation=gravity, store_densities=outputs,
                             store_velocities=outputs)
        s.setFlags(flags, (0, 0, 0), s.size_h)
        s.setDensityDistributions(dd, (0, 0, 0), s.size_h)
        pair.append(s)
    chosen, plain = pair
    for k in (0, 1):
        check(lib().lbm_set_launch_options(plain.handle, k, 0))
    for step in range(4):
        if turns == "round_robin" or (turns == "visits" and step % 2 == 0):
            neighbour.simulationStepAlpha()
        (chosen.simulationStepBeta if step & 1 else chosen.simulationStepAlpha)()
    for step in range(4):
        (plain.simulationStepBeta if step & 1 else plain.simulationStepAlpha)()
    assert np.array_equal(chosen.save_state(), plain.save_state())
    if outputs:
        assert np.array_equal(chosen.getVelocities(), plain.getVelocities())
        assert np.array_equal(chosen.getDensities(), plain.getDensities())
    for s in pair:
        s.close()
