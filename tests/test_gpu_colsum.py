"""Column sums (DGEN_HIP_K_COLSUM) and Adam's one-workgroup form: few rows are
summed in one launch in the two-stage sum's order (bit for bit), a single
column in one workgroup, and the step counter advances once a run whichever
form the update takes.  Needs a GPU."""
import numpy as np
import pytest

from dgen_hip import runtime as R
from dgen_hip.program import Program

pytestmark = pytest.mark.gpu


def colsum(a, cols):
    rows, lda = a.shape
    p = Program(max_frames=1)
    c, o, w = p.alloc("a", rows * lda), p.alloc("o", cols), p.alloc("w", 256 * cols)
    p.add(R.K_COLSUM, [c, o, rows, cols, lda, w])
    with R.HIPLazyRuntime(p) as rt:
        rt.write("a", a)
        for _ in range(2):
            rt.runNoCopy()
        return rt.read("o")


@pytest.mark.parametrize("rows", [9, 31, 63, 64, 65, 250, 511, 512])
@pytest.mark.parametrize("cols", [2, 63, 64, 65, 130])
def test_one_launch_is_the_two_stage_sum(gpu, rows, cols):
    """The same columns inside a matrix wide enough for the two stages."""
    wide = (1 << 19) // rows + 8
    a = np.random.default_rng(rows * cols).standard_normal((rows, wide)).astype(np.float32)
    two = colsum(a, wide)
    np.testing.assert_array_equal(colsum(a, cols), two[:cols])
    ref = a.astype(np.float64).sum(0)
    # pairwise-like order: ~16 + chunks/4 + 6 additions deep
    assert np.abs(two - ref).max() <= 32 * 6e-8 * np.abs(a).sum(0).max()


@pytest.mark.parametrize("at", [0, 1, 70, 130 * 9 + 64])
def test_sum_over_its_source(gpu, at):
    """The result may lie in the summed matrix: the two stages read all of it
    first, and so does a sum that takes one launch elsewhere."""
    rows, cols = 40, 130
    a = np.random.default_rng(at).standard_normal((rows, cols)).astype(np.float32)
    p = Program(max_frames=1)
    c, w = p.alloc("a", rows * cols), p.alloc("w", 256 * cols)
    p.add(R.K_COLSUM, [c, c + at, rows, cols, cols, w])
    print(f"case at={at}", flush=True)
    with R.HIPLazyRuntime(p) as rt:
        rt.write("a", a)
        rt.runNoCopy()
        np.testing.assert_array_equal(rt.read("a")[at:at + cols], colsum(a, cols))


@pytest.mark.parametrize("rows", [1, 1023, 1024, 1025, 16384, 16385])
def test_one_column(gpu, rows):
    a = np.random.default_rng(rows).standard_normal((rows, 1)).astype(np.float32)
    # at most 16 additions in a thread, 6 over the wave, 16 over the waves
    # (one launch), or the two stages' 32 + 128/4
    assert abs(colsum(a, 1)[0] - a.astype(np.float64).sum()) <= 70 * 6e-8 * np.abs(a).sum()


@pytest.mark.parametrize("n", [1, 1000, 4096, 4097])
def test_adam_steps_count_once_a_run(gpu, n):
    rng = np.random.default_rng(n)
    P, G = rng.standard_normal(n).astype(np.float32), rng.standard_normal(n).astype(np.float32)
    p = Program(max_frames=1)
    c = {k: p.alloc(k, s) for k, s in (("p", n), ("g", n), ("m", n), ("v", n), ("t", 1))}
    p.add(R.K_ADAM, [c["p"], c["g"], c["m"], c["v"], n, c["t"]], [1e-2, 0.9, 0.999, 1e-8])
    with R.HIPLazyRuntime(p) as rt:
        rt.write("p", P)
        rt.write("g", G)
        for _ in range(3):
            rt.runNoCopy()
        got, t = rt.read("p"), rt.read("t")[0]
    m, v, ref = np.zeros(n), np.zeros(n), P.astype(np.float64)
    for k in range(1, 4):
        m, v = 0.9 * m + 0.1 * G, 0.999 * v + 0.001 * G.astype(np.float64) ** 2
        ref -= 1e-2 * (m / (1 - 0.9 ** k)) / (np.sqrt(v / (1 - 0.999 ** k)) + 1e-8)
    assert t == 3.0
    # three updates of 1e-2, each within ~1e-4 relative (the fp32 bias
    # corrections 1 - b2^t cancel to ~1e-3), plus the parameter's rounding
    assert np.abs(got - ref).max() <= 3 * 1e-2 * 1e-4 + 2e-7 * np.abs(P).max()
