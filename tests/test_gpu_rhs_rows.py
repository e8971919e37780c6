"""K_rhs's three kernels (tiles of 60 x 16, 60 x 8 and 32 x 26 cells, variants 1,
3 and 5) on fields that are rough everywhere, at the sizes where a tile can go
wrong, with z-chunks of one plane, of unequal depths and of the whole box.  Tiles
of a wave per row: one tile narrower than a wave (32, 36), exactly 60 cells wide
(60, 180), two equal tiles (64, 90, 96), three with a last one narrower (128),
rows that end inside a tile (36, 50, 60, 90, 180).  The flattened 32 x 26 tile:
its smallest box (36), the full width of 32 (64, 96, 128), narrower tiles that
divide the box (36: 18, 60: 30) or not (50: 25 is even, 80: 27, 27, 26), and last
tiles of all but two rows less (128: 24 of 26) down to two rows (80).

phi^{n+1}, v* and P* of one step against the FP64 oracle: a value is the end of
fewer than 400 roundings of terms no larger than the field's largest value
(dt times a stencil stays below it here), so it is off by less than 400 * 2^-24
= 2.4e-5 of that; a missed neighbour is off by 1e-2.  The variants and depths
among each other: bitwise equal."""
import os

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

KEYS = ("h", "dt0", "mu", "cA", "alpha", "beta", "eta", "La", "kappa", "lambda0", "aPhi", "kPhi", "gamma", "A")
BAR = 400 * 2.0 ** -24


@pytest.mark.parametrize("N,A", [(32, 0.0), (36, 0.4), (50, 0.0), (60, 0.4), (64, 0.0), (80, 0.4), (90, 0.4), (96, 0.0), (128, 0.0),
                                 (180, 0.0)])
def test_rough_fields(ttsh, oracle_mod, N, A):
    print(f"[rough_fields N={N}]", flush=True)
    oracle_mod.set_threads(min(16, os.cpu_count() or 1))
    rng = np.random.default_rng(N)
    phi = 0.5 + 0.4 * rng.uniform(-1, 1, (N, N, N))
    P = rng.uniform(-1, 1, (3, N, N, N))
    v = rng.uniform(-1, 1, (3, N, N, N))
    phi, P, v = (x.astype(np.float32).astype(np.float64) for x in (phi, P, v))
    p = ttsh.default_params(N=N, dt0=0.01, A=A, cA=-1.5, La=1.2)
    o = oracle_mod.Oracle(N, faithful=True, **{k: getattr(p, k) for k in KEYS})
    o.set_state(phi, P, v)
    o.step(1)
    want = [o.get_state()[0], o.aux("pstar"), o.aux("vstar")]
    first = None
    for variant, tz in ((1, 7), (3, 7), (1, 1), (3, N), (1, N), (3, 1)) + (((5, 7), (5, 1), (5, N)) if N >= 34 else ()):
        q = p.copy()
        q.rhs_variant, q.rhs_tz = variant, tz
        with ttsh.Simulation(q) as sim:
            sim.set_state(phi, P, v)
            sim.step(1)
            got = [sim.get_state()[0], sim.aux("pstar"), sim.aux("vstar")]
        if first is None:
            first = got
            for name, a, b in zip(("phi", "P*", "v*"), got, want):
                err = float(np.max(np.abs(a - b)) / np.max(np.abs(b)))
                print(f"N={N} {name} {err:.2e}", flush=True)
                assert err <= BAR, name
        else:
            for a, b in zip(got, first):
                assert np.array_equal(a, b), (variant, tz)
