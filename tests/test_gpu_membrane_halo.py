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
    # the gradient's cell terms are summed in fp32 over a launch's steps
    np.testing.assert_allclose(got[3], one[3], rtol=0, atol=8 * 16 * 6e-8 * np.abs(one[2]).max() * np.abs(one[0]).max()
                               * R * C * cfg.T)
