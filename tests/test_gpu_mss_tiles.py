"""Spectral loss (DGEN_HIP_K_SPECTRAL_LOSS): a launch of few tiles transforms
two groups of windows at a time, a larger one a group at a time; both add every
sample in the same order, so a batch row's gradient and window losses do not
depend on how many rows it was run with.  Needs a GPU."""
import numpy as np
import pytest

from dgen_hip import runtime as R
from dgen_hip.program import Program

pytestmark = pytest.mark.gpu
TILE, HALO = 4096, 2047


def mss(x, tgt, sizes, mode):
    B, T = x.shape
    acc = -(-T // TILE) * (TILE + HALO)
    p = Program(max_frames=T)
    cx, ct, cp = p.alloc("x", B * T), p.alloc("tgt", B * T), p.alloc("part", B * acc)
    wl, tabs = [], []
    for n in sizes:
        wl.append(p.alloc(f"wl{n}", -(-T // (n // 4)) * B * 2))
        tabs.append(p.alloc(f"tab{n}", 3 * n - 2))
        p.add(R.K_FFT_TABLES, [tabs[-1], n, 0], flags=R.OP_STATIC)
    pad = lambda v: (list(v) + [0] * 8)[:8]
    p.add(R.K_SPECTRAL_LOSS, [cx, ct, cp, B, T, len(sizes)] + pad(sizes) + pad(wl) + pad(tabs) + [mode], [1e-3, 1e-3])
    with R.HIPLazyRuntime(p) as rt:
        rt.write("x", x)
        rt.write("tgt", tgt)
        rt.runNoCopy()
        return rt.read("part").reshape(B, acc), [rt.read(f"wl{n}").reshape(-1, B, 2) for n in sizes]


@pytest.mark.parametrize("T", [130, 255, 4095, 4097, 9001])
@pytest.mark.parametrize("sizes", [[64, 128, 256, 512, 1024, 2048], [2048, 64]])
@pytest.mark.parametrize("mode", [0, 5])
def test_rows_do_not_depend_on_the_batch(gpu, T, sizes, mode):
    rng = np.random.default_rng(T)
    tiles = -(-T // TILE)
    B = 256 // tiles + 1
    x, tgt = (rng.standard_normal((B, T)).astype(np.float32) for _ in range(2))
    part, wl = mss(x, tgt, sizes, mode)
    few, wlf = mss(x[:3], tgt[:3], sizes, mode)
    np.testing.assert_array_equal(few, part[:3])
    for a, b in zip(wlf, wl):
        np.testing.assert_array_equal(a, b[:, :3])
    assert np.abs(part).max() > 0
