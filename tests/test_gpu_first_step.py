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
