"""K_div's row waves on fields that are rough everywhere, with a previous
predictor that differs from the state, so that every halo position counts: at
sizes of one tile (32, 60), of two and three equal tiles (64, 90, 128), with
rows that end inside a tile (all but 28 n), and z-chunks of one plane, of
unequal depths and of the whole box, in both halo modes.

Pressures (means removed) after one step against the FP64 oracle: the transform
pair rounds about 2 log2(N^3) times, so relative RMS stays below
42 * 2^-24 * 8 = 2e-5 with the packed pair's scale (measured below 1e-6); a
halo cell taken from the wrong step changes p by 1e-2 and more.

The mean of a pressure is the k = 0 coefficient, which only the blocks' FP64 sums
set (k2[0] = 1, so it is minus the mean of s).  A cell's s is the end of fewer
than 32 roundings, so the mean of N^3 of them is off by about 32 * 2^-24 / N^1.5
of their RMS, and that of the pressure, whose transform rounds as often, by as
much of its own; the bar allows ten times both.  A block of b cells left out or
added twice is off by about sqrt(b)/N^3 of the RMS of s: more than 100 times the
bar.  z-chunks of one plane at 128^3 make 3,840 blocks, which k_proj_stats adds;
all others are few enough for the x pass."""
import os

import numpy as np
import pytest

from conftest import rel_rms

pytestmark = pytest.mark.gpu

KEYS = ("h", "dt0", "mu", "cA", "alpha", "beta", "eta", "La", "kappa", "lambda0", "aPhi", "kPhi", "gamma", "A")


def div(u, prev):
    """D.u at h = 1; positions across the periodic boundary read prev, if given."""
    w = [np.pad(p, 1, mode="wrap") for p in (u if prev is None else prev)]
    for a in range(3):
        w[a][1:-1, 1:-1, 1:-1] = u[a]
    cut = lambda f, ax, k: f.take(range(k, f.shape[ax] - 2 + k), ax)
    s = lambda f, ax: (4 * cut(f, ax, 1) + cut(f, ax, 0) + cut(f, ax, 2)) / 6
    d = lambda f, ax: (cut(f, ax, 2) - cut(f, ax, 0)) / 2
    return d(s(s(w[0], 0), 1), 2) + s(d(s(w[1], 0), 1), 2) + s(s(d(w[2], 0), 1), 2)


@pytest.mark.parametrize("N,faithful", [(32, 1), (36, 0), (60, 1), (64, 1), (90, 1), (128, 0), (128, 1)])
def test_rough_fields(ttsh, oracle_mod, N, faithful):
    print(f"[div rough_fields N={N} faithful={faithful}]", flush=True)
    oracle_mod.set_threads(min(16, os.cpu_count() or 1))
    rng = np.random.default_rng(77 + N)
    r = lambda k: rng.uniform(-1, 1, (k, N, N, N)).astype(np.float32).astype(np.float64)
    phi, P, v, vs, ps = 0.5 + 0.4 * r(1)[0], r(3), r(3), r(3), r(3)
    p = ttsh.default_params(N=N, dt0=0.01)
    p.faithful_halo = faithful
    o = oracle_mod.Oracle(N, faithful=bool(faithful), **{k: getattr(p, k) for k in KEYS})
    o.set_state(phi, P, v, vs, ps)
    o.step(1)
    want = [o.aux("p_v"), o.aux("p_p")]
    rms = lambda a: float(np.sqrt((a ** 2).mean()))
    source = [rms(div(o.aux("vstar"), vs if faithful else None) / p.dt0),
              rms(div(o.aux("pstar"), ps if faithful else None) / p.dt0)]
    state = o.get_state()
    for tz in (1, 5, N):
        p.corr_tz = tz
        with ttsh.Simulation(p) as sim:
            sim.set_state(phi, P, v, vs, ps)
            sim.step(1)
            got = sim.aux("p")
            g = sim.get_state()
        for name, a, b in zip(("p_v", "p_p"), got, want):
            err = rel_rms(a - a.mean(), b - b.mean())
            print(f"N={N} tz={tz} {name} {err:.2e}", flush=True)
            assert err <= 2e-5, (name, tz)
        for name, a, b, s in zip(("p_v", "p_p"), got, want, source):
            bar = 320 * 2.0 ** -24 / N ** 1.5 * (s + rms(b))
            print(f"N={N} tz={tz} {name} mean off by {a.mean() - b.mean():.2e}, bar {bar:.2e}", flush=True)
            assert abs(a.mean() - b.mean()) <= bar, (name, tz)
        for a, b in zip(g, state):
            assert rel_rms(a, b) <= 2e-5, tz
