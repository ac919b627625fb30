"""Large host copies whose host side is memory the runtime knows (the device's,
managed, pinned) are the runtime's own, as small ones are."""
import ctypes

import numpy as np
import pytest

from hiprt import DeviceBuffer, rt

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("size", [(30, 20, 10), (101, 99, 97)])   # below and above the ring's
@pytest.mark.parametrize("kind", ["device", "managed", "pinned"])
def test_state_through_memory_the_runtime_knows(hip, kind, size):
    from cavityflow_cuda_amd._lib import check, lib
    print("[case] transfer memory", kind, size, flush=True)
    s = hip.LbmSolverHIP(size)
    s.simulationStepAlpha()
    s.simulationStepBeta()
    s.sync()
    state = s.save_state()
    ptr = ctypes.c_void_p()
    if kind == "device":
        buf = DeviceBuffer(state.size)
        ptr.value = buf.data_ptr()
    elif kind == "managed":
        assert rt().hipMallocManaged(ctypes.byref(ptr), ctypes.c_size_t(state.size), 1) == 0
    else:
        assert rt().hipHostMalloc(ctypes.byref(ptr), ctypes.c_size_t(state.size), 0) == 0
    check(lib().lbm_save_state(s.handle, ptr, ctypes.c_uint64(state.size)))
    check(lib().lbm_reset(s.handle))
    assert not np.array_equal(s.save_state(), state)
    check(lib().lbm_load_state(s.handle, ptr, ctypes.c_uint64(state.size)))
    assert np.array_equal(s.save_state(), state)
    s.close()
    if kind == "device":
        buf.free()
    else:
        assert (rt().hipFree if kind == "managed" else rt().hipHostFree)(ptr) == 0
