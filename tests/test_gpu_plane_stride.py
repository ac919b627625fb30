"""Planes a multiple of 2 MiB apart are moved further apart: the sizes that are,
their bytes, and the results, which a split into other sizes has to repeat."""
import numpy as np
import pytest


def test_bytes_of_padded_planes():
    from cavityflow_cuda_amd.solver import device_bytes
    rest = (1024 + 1) * 5 * 8 + 64
    for size, precision, eb, ob, pad in (((62, 62, 62), "f64", 8, 8, 2304),
                                         ((62, 62, 62), "f32", 4, 4, 0),
                                         ((126, 126, 126), "f16s", 2, 4, 2304),
                                         ((126, 126, 125), "f16s", 2, 4, 0)):
        n = int(np.prod([v + 2 for v in size]))
        stride = (n + 255) // 256 * 256 + pad
        assert device_bytes(size, precision) == 19 * stride * eb + stride + rest + 3 * stride * ob


@pytest.mark.gpu
@pytest.mark.parametrize("precision,size", [("f64", (62, 62, 62)), ("f32", (126, 62, 62)),
                                            ("f16s", (126, 126, 126)), ("f16c", (254, 62, 62))])
def test_padded_planes_keep_the_bits(hip, precision, size):
    from cavityflow_cuda_amd.controller import CavityController
    print("[case] plane stride", precision, size, flush=True)
    fields = []
    for split in ((1, 1, 1), (2, 1, 1)):
        c = CavityController(size, 0.05, 100.0, precision, split=split)
        for s in c.solvers.values():
            a = s.device_arrays()
            cells = int(np.prod(s.size_h))
            assert a.plane_stride % 256 == 0 and a.plane_stride >= cells
            assert (a.plane_stride - cells >= 2304) == (split == (1, 1, 1))
        for _ in range(4):
            c.computeNextStep()
        c.sync()
        fields.append((c.getVelocities(), c.getDensities()))
        if split == (1, 1, 1):
            s = c.solvers[(0, 0, 0)]
            saved = s.save_state()
            s.load_state(saved)
            assert np.array_equal(saved, s.save_state())
        c.close()
    assert np.array_equal(fields[0][0], fields[1][0])
    assert np.array_equal(fields[0][1], fields[1][1])
