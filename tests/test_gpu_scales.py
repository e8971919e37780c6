"""The stencils' scale s = 1/(72 h) is rounded once, from FP64, and the
divergence's s/dt0 is its product with 1/dt0.

K_rhs: phi is 0 on every second cell (a checkerboard) and a small whole number on
the others, v = (1, 0, 0), gamma = 0, Dt = 2^-7.  At the zeros phi^{n+1} is then
-Dt fl(s d), d a whole number (the raw stencil's sum), which FP32 gives exactly:
bitwise equal.  At h = 0.93 and 1.49 fl(fl(1/2h) fl(1/36)) is another number.

K_div: p of one step against the FP64 oracle, as the ratio of the two fields, in
which the roundings of 32^3 cells average out (2e-7/sqrt(32^3) = 1e-9).  What is
left is the rounding of s/dt0 and of the Poisson factor's constant, both known,
and that of the transform's constants, the same for every h.  At h = 1.377,
dt0 = 0.006 the first two are -1e-8 together, where a product of three rounded
factors, 1/(2h), 1/36 and 1/dt0, makes 1.3e-7; so the difference to h = 1,
dt0 = 1/128, where either product rounds as once, tells them apart, with a bar of
3e-8."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

F = np.float32
OFF = dict(mu=0.0, cA=0.0, alpha=0.0, beta=0.0, eta=0.0, lambda0=0.0, aPhi=0.0, kPhi=0.0, gamma=0.0, A=0.0)


def raw_dx(f):
    """72 h D_x f: [1,4,1] over z and y, [-1,0,1] over x."""
    s = lambda a, ax: 4 * a + np.roll(a, 1, ax) + np.roll(a, -1, ax)
    g = s(s(f, 0), 1)
    return np.roll(g, -1, 2) - np.roll(g, 1, 2)


@pytest.mark.parametrize("variant", [1, 3, 5])
@pytest.mark.parametrize("h", [0.93, 1.49])
def test_rhs_scale(ttsh, h, variant):
    print(f"[rhs_scale h={h} variant={variant}]", flush=True)
    N, Dt = 64, 2.0 ** -7
    s = F(1.0 / (72.0 * h))
    assert F(F(1.0 / (2.0 * h)) * F(F(1) / F(36))) != s
    rng = np.random.default_rng(8)
    z, y, x = np.indices((N, N, N))
    zero = (x + y + z) % 2 == 0
    phi = np.where(zero, 0, rng.integers(-3, 4, (N, N, N))).astype(np.int64)
    v = np.zeros((3, N, N, N), F)
    v[0] = 1
    p = ttsh.default_params(N=N, dt0=Dt, h=h, **OFF)
    p.rhs_variant = variant
    with ttsh.Simulation(p) as sim:
        sim.set_state(phi.astype(F), np.zeros_like(v), v, dtype=ttsh.F32)
        sim.step(1)
        got = sim.get_state()[0]
    want = -F(Dt) * (s * raw_dx(phi).astype(F))
    assert np.array_equal(got[zero], want[zero])


def scale_rounding(N, h, dt):
    """Relative roundings of s/dt0 and of -1/((2 pi/(N h))^2 N^3), added."""
    off = lambda a, b: float(a) / b - 1.0
    k = -1.0 / ((2.0 * np.pi / (N * h)) ** 2 * N ** 3)
    return off(F(1.0 / (72.0 * h)) * F(1.0 / dt), 1.0 / (72.0 * h * dt)) + off(F(k), k)


def test_div_scale(ttsh, oracle_mod):
    print("[div_scale]", flush=True)
    N = 32
    rng = np.random.default_rng(9)
    r = lambda k: rng.uniform(-1, 1, (k, N, N, N)).astype(F)
    phi, P, v = np.zeros((N, N, N)), r(3).astype(np.float64), (F(1e-3) * r(3)).astype(np.float64)
    left = []
    for h, dt in ((1.377, 0.006), (1.0, 2.0 ** -7)):
        par = dict(h=h, dt0=dt, La=1.0, kappa=0.0, **OFF)
        p = ttsh.default_params(N=N, **par)
        p.faithful_halo = 0
        o = oracle_mod.Oracle(N, faithful=False, **par)
        o.set_state(phi, P, v)
        o.step(1)
        with ttsh.Simulation(p) as sim:
            sim.set_state(phi, P, v)
            sim.step(1)
            got = sim.aux("p")
        for name, a, b in zip(("p_v", "p_p"), got, (o.aux("p_v"), o.aux("p_p"))):
            a, b = a - a.mean(), b - b.mean()
            left.append(float((a * b).sum() / (b * b).sum()) - 1.0 - scale_rounding(N, h, dt))
            print(f"h={h} {name}: {left[-1]:.2e} beside the scales' roundings", flush=True)
    for a, b in zip(left[:2], left[2:]):
        assert abs(a - b) < 3e-8
