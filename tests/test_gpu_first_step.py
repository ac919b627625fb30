"""A solver's first half-steps are launched as its later ones in the same state of
the caches: the choice follows the bytes stepped in between, not how often the
solver has been stepped."""
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision,size", [("f32", (20, 16, 12)), ("f32", (229, 186, 141)),
                                            ("f32", (150, 150, 150)), ("f64", (160, 150, 140)),
                                            ("f16s", (190, 187, 193))])
def test_first_steps_are_launched_as_later_ones(hip, precision, size):
    from hiprt import stream_create, stream_destroy
    from launches import launches
    print("[case] first step", precision, size, flush=True)
    s = hip.LbmSolverHIP(size, precision=precision, store_densities=False,
                         store_velocities=False)
    st = stream_create()
    seen = [(launches(lambda h: s.simulationStepAlpha(stream=h), st),
             launches(lambda h: s.simulationStepBeta(stream=h), st)) for _ in range(3)]
    stream_destroy(st)
    s.close()
    assert all(len(a) == 1 and len(b) == 1 for a, b in seen)
    assert seen[0] == seen[1] == seen[2]


def test_first_steps_of_solvers_that_do_not_fit_together(hip):
    """Eight solvers that fit the Infinity Cache each but not together, every state
    written after the others' creation: alpha finds nothing of its state in the cache
    and streams, so beta finds nothing either, also right after it."""
    from cavityflow_cuda_amd._lib import check, lib
    from hiprt import stream_create, stream_destroy
    from launches import launches
    print("[case] first steps of eight", flush=True)
    NT, W2 = 1, 16
    solvers = [hip.LbmSolverHIP((100, 99, 98), store_densities=False, store_velocities=False)
               for _ in range(9)]
    named = solvers.pop()
    for k, options in ((0, NT | W2), (1, W2)):
        check(lib().lbm_set_launch_options(named.handle, k, options))
    for s in solvers:
        s.setDensityDistributions(s.getDensityDistributions())
    st = stream_create()
    alpha = [launches(lambda h: s.simulationStepAlpha(stream=h), st) for s in solvers]
    beta = [launches(lambda h: s.simulationStepBeta(stream=h), st) for s in reversed(solvers)]
    assert alpha == [launches(lambda h: named.simulationStepAlpha(stream=h), st)] * 8
    assert beta == [launches(lambda h: named.simulationStepBeta(stream=h), st)] * 8
    stream_destroy(st)
    for s in solvers + [named]:
        s.close()
