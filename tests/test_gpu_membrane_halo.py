"""2D membrane: the waves of a launch's halo leave once their rows can no
longer reach the tile, so launches of any number of steps (and regions inside
the grid, at its edges or centred over a small one) give the same states and
adjoint fields, bit for bit.  Needs a GPU."""
import numpy as np
import pytest

from dgen_hip import MembraneConfig
from dgen_hip.programs import membrane_program
from dgen_hip.runtime import HIPLazyRuntime

pytestmark = pytest.mark.gpu


def run(cfg, u0, tgt, steps):
    with HIPLazyRuntime(membrane_program(cfg, train=True, steps=steps), 0) as rt:
        rt.write("u0", u0)
        rt.write("params", cfg.params())
        rt.write("target", tgt)
        rt.runNoCopy()
        last = (-(-(cfg.T + 1) // steps) - 1) % 2  # the adjoint set of the last launch
        return (rt.read("states"), rt.read("pickup"), rt.read("adjoint_fields").reshape(2, -1)[last],
                rt.read("grads"))


def lap(u, centre=-4.0):
    p = np.pad(u, 1)
    return p[:-2, 1:-1] + p[2:, 1:-1] + p[1:-1, :-2] + p[1:-1, 2:] + centre * u


def gradient64(cfg, u0, tgt):
    """(d/dc2, d/dd) in fp64 and the sums of their terms' magnitudes."""
    c2, d = (float(v) for v in cfg.params())
    u = [u0.astype(np.float64)] * 2  # u_{-1}, u_0, ...
    for _ in range(cfg.T):
        u.append(2 * u[-1] - u[-2] + c2 * lap(u[-1]) - d * (u[-1] - u[-2]))
    l1, l2 = np.zeros_like(u[0]), np.zeros_like(u[0])
    g, mag = np.zeros(2), np.zeros(2)
    for n in range(cfg.T, 0, -1):
        lam = (2 - d) * l1 + c2 * lap(l1) - (1 - d) * l2
        lam[cfg.pickup] += 2 * (u[n + 1][cfg.pickup] - tgt[n - 1])
        v, w = u[n], u[n - 1]  # u_{n-1}, u_{n-2}
        g += [(lam * lap(v)).sum(), (lam * (w - v)).sum()]
        mag += [(abs(lam) * lap(abs(v), 4.0)).sum(), (abs(lam) * (abs(w) + abs(v))).sum()]
        l1, l2 = lam, l1
    return g, mag


@pytest.mark.parametrize("R,C", [(64, 64), (33, 200), (97, 65), (160, 31), (5, 3)])
@pytest.mark.parametrize("steps", [2, 5, 12, 13, 16])
def test_steps_per_launch_do_not_change_the_fields(gpu, R, C, steps):
    cfg = MembraneConfig(R=R, C=C, T=39)
    rng = np.random.default_rng(R)
    u0 = rng.standard_normal((R, C)).astype(np.float32)  # every cell matters
    tgt = rng.standard_normal(cfg.T).astype(np.float32)
    one = run(cfg, u0, tgt, 1)
    got = run(cfg, u0, tgt, steps)
    for a, b in zip(got[:3], one[:3]):
        np.testing.assert_array_equal(a, b)
    # fp32 states, adjoint and per-launch sums, roundings of either sign in
    # every one of the terms: 16 half ulps of the terms' magnitudes in all (the
    # fp32 oracle stays within 0.7 of one)
    g64, mag = gradient64(cfg, u0, tgt)
    print(f"gradient {got[3]} fp64 {g64} terms {mag}", flush=True)
    assert (np.abs(got[3] - g64) <= 16 * 2.0**-24 * mag).all()
    assert (np.abs(one[3] - g64) <= 16 * 2.0**-24 * mag).all()
