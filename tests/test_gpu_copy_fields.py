"""ttsh_step_noalloc copies a state in and out with one kernel each, 16 bytes at
a time where every array begins on a 16-byte boundary and 4 otherwise.  Caller
arrays at offsets of 0 to 3 floats: the state and predictors equal ttsh_step's
bitwise, and the floats around each array stay as they were."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,offset", [(32, 0), (32, 1), (36, 2), (50, 3), (64, 0), (64, 1)])
def test_offsets(ttsh, N, offset):
    import torch
    print(f"[copy_fields N={N} offset={offset}]", flush=True)
    rng = np.random.default_rng(N + offset)
    r = lambda k: rng.uniform(-1, 1, (k, N, N, N)).astype(np.float32)
    state = (0.5 + 0.4 * r(1)[0], r(3), 0.1 * r(3))
    prev = (0.1 * r(3), r(3))
    p = ttsh.default_params(N=N, dt0=0.005)
    held = []
    for a in (*state, *prev):
        t = torch.full((a.size + 8,), 7.0, device="cuda")
        t[4 + offset:4 + offset + a.size] = torch.from_numpy(a.reshape(-1)).cuda()
        held.append((t, a.size))
    torch.cuda.synchronize()
    ttsh.step_noalloc(p, *(t.data_ptr() + 4 * (4 + offset) for t, _ in held), 3)
    with ttsh.Simulation(p) as s:
        s.set_state(*state, *prev, dtype=ttsh.F32)
        s.step(3)
        want = (*s.get_state(), s.aux("vstar"), s.aux("pstar"))
    for (t, n), b in zip(held, want):
        got = t.cpu().numpy()
        assert np.array_equal(got[4 + offset:4 + offset + n], b.reshape(-1))
        assert (got[:4 + offset] == 7.0).all() and (got[4 + offset + n:] == 7.0).all()
