"""Batches of several sizes run one FFT launch per pass for all of them
(k_fft_sizes) and cut K_rhs, K_div and K_corr into chunks of one depth for the
whole batch.  Every planned size, in three batches of one droplet per size:
each droplet equals its run alone bitwise, with plain launches and, for the
small sizes, with graph replay.  The states are rough everywhere, so that a
line or plane left out shows.

And a graph batch whose FFT launches change between replays, as its droplets
reach their limits one by one."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def state(N, seed):
    rng = np.random.default_rng(seed)
    r = lambda k: (2.0 * rng.random((k, N, N, N), dtype=np.float32) - 1.0)
    return 0.5 + 0.4 * r(1)[0], r(3), 0.1 * r(3)


@pytest.mark.parametrize("sizes,steps,graph", [
    ((32, 36, 40, 48, 50, 60, 64, 72), 19, True),
    ((80, 90, 96, 100, 120, 128, 144, 150), 2, False),
    ((160, 180, 192, 200, 240, 256), 1, False)])
def test_every_size_in_a_batch_equals_alone(ttsh, sizes, steps, graph):
    print(f"[every_size_in_a_batch_equals_alone {sizes}]", flush=True)
    params = [ttsh.default_params(N=N, dt0=0.005, cA=-1.0 - 0.1 * k) for k, N in enumerate(sizes)]
    with ttsh.Batch(max_slots=len(sizes), use_graph=graph) as b:
        slots = [b.admit(p, *state(p.Nx, 900 + p.Nx), dtype=ttsh.F32) for p in params]
        b.step(steps)
        got = [b.get_state(s) for s in slots]
    for p, g in zip(params, got):
        print(f"N={p.Nx}", flush=True)
        with ttsh.Simulation(p) as sim:
            sim.set_state(*state(p.Nx, 900 + p.Nx), dtype=ttsh.F32)
            sim.step(steps)
            ref = sim.get_state()
        assert all(np.isfinite(x).all() for x in ref)
        for x, y in zip(ref, g):
            assert np.array_equal(x, y), f"N={p.Nx}"


def test_graph_replays_while_the_fft_launches_change(ttsh):
    """144^3, 150^3, 96^3 and 80^3 in one graph batch: at first shared launches
    for the x passes, for the y and z passes of the large sizes and for the
    planes of the small ones; without 144^3 a y and z pass of one size; without
    150^3 an x pass that adds up the projection's sums (976 groups on 256 CUs);
    without 96^3 a launch per pass of one size.  Each layout is replayed, from
    either parity, and each droplet equals its run alone bitwise."""
    print("[graph_replays_while_the_fft_launches_change]", flush=True)
    limits = {144: 20, 150: 52, 96: 101, 80: 139}
    params = {N: ttsh.default_params(N=N, dt0=0.005, cA=-1.2) for N in limits}
    with ttsh.Batch(max_slots=4, use_graph=True) as b:
        slots = {N: b.admit(params[N], *state(N, 50 + N), dtype=ttsh.F32, limit=limits[N]) for N in limits}
        for n in (33, 35, 33, 39):
            b.step(n)
        assert all(b.steps_done(slots[N]) == limits[N] for N in limits)
        got = {N: b.get_state(slots[N]) for N in limits}
    for N, steps in limits.items():
        print(f"N={N}", flush=True)
        with ttsh.Simulation(params[N]) as sim:
            sim.set_state(*state(N, 50 + N), dtype=ttsh.F32)
            sim.step(steps)
            ref = sim.get_state()
        assert all(np.isfinite(x).all() for x in ref)
        for x, y in zip(ref, got[N]):
            assert np.array_equal(x, y), f"N={N}"
