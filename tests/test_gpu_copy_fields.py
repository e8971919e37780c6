"""ttsh_step_noalloc copies a state in and out with one kernel each, 16 bytes at
a time where every array begins on a 16-byte boundary and 4 otherwise.  Caller
arrays at offsets of 0 to 3 floats: the state and predictors equal ttsh_step's
bitwise, and the floats around each array stay as they were.  Device memory
comes from the HIP runtime that the library itself loads, through ctypes."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

H2D, D2H = 1, 2  # hipMemcpyHostToDevice, hipMemcpyDeviceToHost


@pytest.mark.parametrize("N,offset", [(32, 0), (32, 1), (36, 2), (50, 3), (64, 0), (64, 1)])
def test_offsets(ttsh, N, offset):
    print(f"[copy_fields N={N} offset={offset}]", flush=True)
    ttsh.lib()
    hip = ctypes.CDLL("libamdhip64.so.7")
    hip.hipMalloc.argtypes = [ctypes.POINTER(ctypes.c_void_p), ctypes.c_size_t]
    hip.hipFree.argtypes = [ctypes.c_void_p]
    hip.hipMemcpy.argtypes = [ctypes.c_void_p, ctypes.c_void_p, ctypes.c_size_t, ctypes.c_int]
    rng = np.random.default_rng(N + offset)
    r = lambda k: rng.uniform(-1, 1, (k, N, N, N)).astype(np.float32)
    state = (0.5 + 0.4 * r(1)[0], r(3), 0.1 * r(3))
    prev = (0.1 * r(3), r(3))
    p = ttsh.default_params(N=N, dt0=0.005)
    begin = 4 + offset
    held = []
    try:
        for a in (*state, *prev):
            host = np.full(a.size + 8, 7.0, np.float32)
            host[begin:begin + a.size] = a.reshape(-1)
            ptr = ctypes.c_void_p()
            assert hip.hipMalloc(ctypes.byref(ptr), host.nbytes) == 0
            held.append((ptr, host))
            assert hip.hipMemcpy(ptr, host.ctypes.data, host.nbytes, H2D) == 0
        assert hip.hipDeviceSynchronize() == 0
        ttsh.step_noalloc(p, *(ptr.value + 4 * begin for ptr, _ in held), 3)
        for ptr, host in held:
            assert hip.hipMemcpy(host.ctypes.data, ptr, host.nbytes, D2H) == 0
    finally:
        for ptr, _ in held:
            hip.hipFree(ptr)
    with ttsh.Simulation(p) as s:
        s.set_state(*state, *prev, dtype=ttsh.F32)
        s.step(3)
        want = (*s.get_state(), s.aux("vstar"), s.aux("pstar"))
    for (_, got), b in zip(held, want):
        assert np.array_equal(got[begin:begin + b.size], b.reshape(-1))
        assert (got[:begin] == 7.0).all() and (got[begin + b.size:] == 7.0).all()


@pytest.mark.parametrize("memory", ["pageable", "pinned", "phi pageable", "v* is v"])
def test_memory_that_the_copy_kernel_may_not_touch(ttsh, memory):
    """Host arrays, and arrays of which two are the same memory, take the
    runtime's copies: a kernel would fault on the first and write the second in
    no order.  The state equals ttsh_step's bitwise; of one array given twice
    the later copy, the predictor, is what remains."""
    print(f"[copy_fields {memory}]", flush=True)
    ttsh.lib()
    hip = ctypes.CDLL("libamdhip64.so.7")
    hip.hipMalloc.argtypes = [ctypes.POINTER(ctypes.c_void_p), ctypes.c_size_t]
    hip.hipHostMalloc.argtypes = [ctypes.POINTER(ctypes.c_void_p), ctypes.c_size_t, ctypes.c_uint]
    hip.hipFree.argtypes = hip.hipHostFree.argtypes = [ctypes.c_void_p]
    hip.hipMemcpy.argtypes = [ctypes.c_void_p, ctypes.c_void_p, ctypes.c_size_t, ctypes.c_int]
    N = 36
    rng = np.random.default_rng(5)
    r = lambda k: rng.uniform(-1, 1, (k, N, N, N)).astype(np.float32)
    phi, P, v = 0.5 + 0.4 * r(1)[0], r(3), 0.1 * r(3)
    p = ttsh.default_params(N=N, dt0=0.005)
    begin = [phi, P, v, v.copy(), P.copy()]
    out = [a.copy() for a in begin]
    ptrs, frees = [], []
    try:
        for k, a in enumerate(out):
            ptr = ctypes.c_void_p()
            if memory == "pageable" or (memory == "phi pageable" and k == 0):
                ptr.value = a.ctypes.data
            elif memory == "pinned":
                assert hip.hipHostMalloc(ctypes.byref(ptr), a.nbytes, 0) == 0
                frees.append((hip.hipHostFree, ptr))
                ctypes.memmove(ptr, a.ctypes.data, a.nbytes)
                out[k] = np.ctypeslib.as_array((ctypes.c_float * a.size).from_address(ptr.value))
            else:
                assert hip.hipMalloc(ctypes.byref(ptr), a.nbytes) == 0
                frees.append((hip.hipFree, ptr))
                assert hip.hipMemcpy(ptr, a.ctypes.data, a.nbytes, H2D) == 0
                out[k] = None
            ptrs.append(ptr)
        if memory == "v* is v":
            ptrs[3] = ptrs[2]
        assert hip.hipDeviceSynchronize() == 0
        ttsh.step_noalloc(p, *(q.value for q in ptrs), 3)
        got = []
        for q, a, b in zip(ptrs, out, begin):
            if a is None:
                a = np.empty(b.size, np.float32)
                assert hip.hipMemcpy(a.ctypes.data, q, a.nbytes, D2H) == 0
            got.append(a.reshape(-1).copy())
    finally:
        for free, q in frees:
            free(q)
    with ttsh.Simulation(p) as s:
        s.set_state(*begin, dtype=ttsh.F32)
        s.step(3)
        want = [x.reshape(-1) for x in (*s.get_state(), s.aux("vstar"), s.aux("pstar"))]
    if memory == "v* is v":
        want[2] = want[3]
    for a, b in zip(got, want):
        assert np.array_equal(a, b)
