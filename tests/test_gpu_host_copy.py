"""State out to host arrays: the plain copy (small boxes) and the chunked one
with worker threads (8 MiB of state and more), in FP32 and FP64, at sizes whose
fields end inside a 4 MiB chunk, just above one and far below; from two handles
on two threads at once.  What went in comes out bit for bit."""
import ctypes
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def state(N, seed):
    rng = np.random.default_rng(seed)
    r = lambda k: rng.random((k, N, N, N), dtype=np.float32)
    return r(1)[0], r(3), r(3)


def round_trip(ttsh, N, seed):
    st = state(N, seed)
    with ttsh.Simulation(ttsh.default_params(N=N)) as sim:
        sim.set_state(*st, dtype=ttsh.F32)
        for dtype in (ttsh.F32, ttsh.F64, ttsh.F32):
            for a, b in zip(st, sim.get_state(dtype)):
                assert b.dtype == (np.float32 if dtype == ttsh.F32 else np.float64)
                assert np.array_equal(a, b), (N, dtype)


@pytest.mark.parametrize("N", [32, 64, 72, 100, 120, 160])
def test_round_trip(ttsh, N):
    print(f"[round_trip N={N}]", flush=True)
    round_trip(ttsh, N, N)


def test_two_threads(ttsh):
    print("[two_threads]", flush=True)
    failed = []

    def go(seed):
        try:
            for k in range(3):
                round_trip(ttsh, 100, seed + k)
        except Exception as e:  # noqa: BLE001
            failed.append(e)

    ts = [threading.Thread(target=go, args=(10 * k,)) for k in range(2)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert not failed


@pytest.mark.parametrize("f64", [False, True])
def test_pinned_destination(ttsh, f64):
    """phi in pinned memory (FP32: a copy of its own, without the chunks), P and
    v in pageable memory."""
    print(f"[pinned_destination f64={f64}]", flush=True)
    N = 100
    st = state(N, 5)
    t, dtype = (np.float64, ttsh.F64) if f64 else (np.float32, ttsh.F32)
    hip = ctypes.CDLL("libamdhip64.so.7")
    hip.hipHostMalloc.argtypes = [ctypes.POINTER(ctypes.c_void_p), ctypes.c_size_t, ctypes.c_uint]
    hip.hipHostFree.argtypes = [ctypes.c_void_p]
    P, v = np.empty((3, N, N, N), t), np.empty((3, N, N, N), t)
    at = lambda a: a.ctypes.data_as(ctypes.c_void_p)
    with ttsh.Simulation(ttsh.default_params(N=N)) as sim:
        sim.set_state(*st, dtype=ttsh.F32)
        pin = ctypes.c_void_p()
        assert hip.hipHostMalloc(ctypes.byref(pin), P.nbytes // 3, 0) == 0
        try:
            assert ttsh.lib().ttsh_get_state(sim._h, dtype, pin, at(P), at(v)) == 0
            phi = np.frombuffer((ctypes.c_char * (P.nbytes // 3)).from_address(pin.value), t).reshape(N, N, N).copy()
        finally:
            hip.hipHostFree(pin)
    for a, b in zip(st, (phi, P, v)):
        assert np.array_equal(a, b)
