"""Host copies of every size class: below the pinned ring, one chunk, several
with a remainder, planes that are not multiples of a chunk; two threads at
once; numpy arrays and pinned memory. What comes back is what went in."""
import ctypes
import threading

import numpy as np
import pytest

from hiprt import rt

pytestmark = pytest.mark.gpu


def filled(hip, precision, size, seed):
    s = hip.LbmSolverHIP(size, precision=precision)
    rng = np.random.default_rng(seed)
    state = s.save_state()
    n = int(np.prod(s.size_h))
    width = {"f32": 4, "f64": 8, "f16s": 2}[precision]
    dtype = {"f32": np.float32, "f64": np.float64, "f16s": np.float16}[precision]
    state[:19 * n * width] = rng.uniform(0.01, 0.3, 19 * n).astype(dtype).view(np.uint8)
    return s, state


@pytest.mark.parametrize("precision,size", [
    ("f32", (7, 5, 3)), ("f32", (62, 40, 38)), ("f64", (53, 50, 49)), ("f32", (101, 99, 97)),
    ("f16s", (130, 64, 67)), ("f64", (150, 81, 61))])
def test_state_and_fields_round_trip(hip, precision, size):
    print("[case] host transfer", precision, size, flush=True)
    s, state = filled(hip, precision, size, 9)
    s.load_state(state)
    assert np.array_equal(s.save_state(), state)
    rng = np.random.default_rng(4)
    full = ((0, 0, 0), s.size_h)
    n = int(np.prod(s.size_h))
    u, rho = rng.random(3 * n).astype(s.dtype), rng.random(n).astype(s.dtype)
    flags = rng.choice(np.array([1, 2, 4, 8], np.int32), n)
    s.setVelocities(u, *full)
    s.setDensities(rho, *full)
    s.setFlags(flags, *full)
    assert np.array_equal(s.getVelocities(*full), u)
    assert np.array_equal(s.getDensities(*full), rho)
    assert np.array_equal(s.getFlags(*full), flags)
    if precision != "f16s":
        f = rng.uniform(0.01, 0.3, 19 * n).astype(s.dtype)
        s.setDensityDistributions(f, *full)
        assert np.array_equal(s.getDensityDistributions(*full), f)
    s.close()


def test_two_threads_and_pinned_memory(hip):
    print("[case] host transfer threads", flush=True)
    pairs = [filled(hip, "f32", (80, 70 + 3 * k, 60), k) for k in range(2)]
    bad = []

    def work(s, state):
        for _ in range(4):
            s.load_state(state)
            if not np.array_equal(s.save_state(), state):
                bad.append(s)

    threads = [threading.Thread(target=work, args=p) for p in pairs]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad
    s, state = pairs[0]
    ptr = ctypes.c_void_p()
    assert rt().hipHostMalloc(ctypes.byref(ptr), ctypes.c_size_t(state.size), 0) == 0
    pinned = np.ctypeslib.as_array(ctypes.cast(ptr, ctypes.POINTER(ctypes.c_uint8)), (state.size,))
    pinned[:] = state[::-1]
    pinned[-int(np.prod(s.size_h)):] = 2   # flags
    s.load_state(pinned)
    assert np.array_equal(s.save_state(), pinned)
    for s, _ in pairs:
        s.close()
    assert rt().hipHostFree(ptr) == 0
