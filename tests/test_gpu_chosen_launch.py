"""What whole-domain steps launch when their options were not set: the kernel, the
workgroups and the cap on the waves of the options that the choice names for the
size (those a caller can set; the order of the cells is an argument), pairs of cells
for the 16-bit formats; and the bits of plain launches."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

X, W4, W2, LDS, BIG = 2, 4, 16, 128, 256
# precision, interior size, alpha and beta options; None: pairs of cells
ROWS = [("f32", (20, 16, 12), 0, 0), ("f32", (37, 33, 31), X, X), ("f32", (62, 62, 62), X, X),
        ("f32", (62, 30, 62), X, X), ("f32", (86, 83, 81), 0, X | W2),
        ("f32", (151, 149, 150), W4, BIG | W4), ("f64", (37, 33, 31), X, X),
        ("f64", (150, 147, 139), W2, W2), ("f64", (233, 232, 231), W2, LDS | W2),
        ("f16s", (107, 103, 101), None, None), ("f16c", (190, 187, 193), None, None)]


@pytest.mark.parametrize("precision,size,alpha,beta", ROWS)
def test_chosen_launch(hip, precision, size, alpha, beta):
    from cavityflow_cuda_amd._lib import check, lib
    from hiprt import stream_create, stream_destroy
    from launches import launches
    print("[case] chosen launch", precision, size, flush=True)
    named, plain, chosen = (hip.LbmSolverHIP(size, precision=precision, inv_tau=1.3,
                                             lid_velocity=0.07, store_densities=False,
                                             store_velocities=False) for _ in range(3))
    st = stream_create()
    for k, options in ((0, alpha), (1, beta)):
        check(lib().lbm_set_launch_options(named.handle, k, options or 0))
        check(lib().lbm_set_launch_options(plain.handle, k, 0))
    seen = []
    for s in (chosen, named):   # nothing between the creation of `chosen` and its steps
        seen.append(launches(lambda h: s.simulationStepAlpha(stream=h), st) +
                    launches(lambda h: s.simulationStepBeta(stream=h), st))
    if alpha is None:
        n = int(np.prod([v + 2 for v in size]))
        assert [x[1:3] for x in seen[0]] == [((-(-n // 512), 1, 1), (256, 1, 1))] * 2
        assert all(a[0] != b[0] for a, b in zip(*seen))
    else:
        assert seen[0] == seen[1]
    for s in (chosen, plain):
        s.setDrivenCavitySzenario()
        for step in range(6):
            (s.simulationStepBeta if step & 1 else s.simulationStepAlpha)()
    assert np.array_equal(chosen.save_state(), plain.save_state())
    for s in (chosen, named, plain):
        s.close()
    stream_destroy(st)
