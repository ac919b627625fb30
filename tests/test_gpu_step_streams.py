"""Whole-domain steps on several streams: received faces unpacked beside an alpha of
the same solver, and several solvers stepped side by side, give the bits of the same
calls one after the other."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def solver(hip, precision, size, bc, seed):
    s = hip.LbmSolverHIP(size, bc, precision, 1.3, 0.07, store_densities=False,
                         store_velocities=False)
    w = np.array([1 / 18] * 4 + [1 / 36] * 12 + [1 / 18] * 2 + [1 / 3])
    n = int(np.prod(s.size_h))
    noise = np.random.default_rng(seed).uniform(0.97, 1.03, n)
    s.setDensityDistributions((w[:, None] * noise[None, :]).astype(s.dtype).ravel(), (0, 0, 0),
                              s.size_h)
    return s


@pytest.mark.parametrize("precision,size", [("f16s", (126, 103, 101)), ("f16c", (127, 103, 101)),
                                            ("bf16s", (190, 187, 193)), ("f32", (126, 103, 101))])
def test_faces_unpacked_beside_alpha(hip, precision, size):
    """GHOST_LAYER faces; an even and odd number of cells in a row, so that ghosts share
    words with the cells beside them."""
    from hiprt import DeviceBuffer, stream_create, stream_destroy
    print("[case] unpack beside alpha", precision, size, flush=True)
    beside, after = (solver(hip, precision, size, (8,) * 6, 3) for _ in range(2))
    streams = [stream_create(), stream_create()]
    rng = np.random.default_rng(5)
    width = np.dtype(beside.dtype).itemsize
    for step in range(4):
        faces = []
        for d in range(6):
            n = beside.face_elements(d)
            faces.append(DeviceBuffer(n * width))
            faces[d].upload(rng.uniform(0.02, 0.06, n).astype(beside.dtype))
        beside.simulationStepAlpha(stream=streams[0])
        for d in range(6):
            beside.unpack_face(d, 0, faces[d], stream=streams[1])
        after.simulationStepAlpha()
        after.sync()
        for d in range(6):
            after.unpack_face(d, 0, faces[d])
        for st in streams:
            beside.sync(st)
        assert np.array_equal(beside.save_state(), after.save_state()), step
        for s in (beside, after):
            s.simulationStepBeta()
            s.sync()
    for s in (beside, after):
        s.close()
    for st in streams:
        stream_destroy(st)


def test_solvers_side_by_side(hip):
    from hiprt import stream_create, stream_destroy
    print("[case] solvers side by side", flush=True)
    cases = [("f32", (86, 83, 81)), ("f16s", (107, 103, 101)), ("f64", (90, 84, 81)),
             ("f16c", (150, 149, 147))]
    for turns in (1, 6):
        got, streams = [], [stream_create() for _ in cases]
        for own in (True, False):
            solvers = [solver(hip, p, size, (1,) * 6, 7) for p, size in cases]
            for step in range(0, 6, turns):
                for s, st in zip(solvers, streams if own else [None] * len(cases)):
                    for k in range(step, step + turns):
                        (s.simulationStepBeta if k & 1 else s.simulationStepAlpha)(stream=st)
            for s, st in zip(solvers, streams if own else [None] * len(cases)):
                s.sync(st)
            got.append([s.save_state() for s in solvers])
            for s in solvers:
                s.close()
        assert all(np.array_equal(a, b) for a, b in zip(*got))
        for st in streams:
            stream_destroy(st)
