"""Temporal gradient of stateful accumulators on the GPU: the chunked
reset-aware suffix scan (DGEN_HIP_K_TEMPORAL_GRAD_SCAN) against the oracle's
sequential scan (Emit+TemporalGradient.swift:56-81), and the swept-phasor
bank's gradient to its learnable sweep rates against the fp64 oracle and
central finite differences of it (TemporalGradientTests.swift:24-60 scaled
to 256 lanes x 2^16 frames).  Needs a GPU."""
import numpy as np
import pytest

import oracle as O
from dgen_hip import SweptPhasorConfig
from dgen_hip import runtime as R
from dgen_hip.program import Program
from dgen_hip.programs import SweptPhasorSession

pytestmark = pytest.mark.gpu


def scan_program(E, T):
    p = Program(max_frames=T)
    g = p.alloc("g", T * E)
    rs = p.alloc("reset", T)
    out = p.alloc("out", T * E)
    C = (T + 255) // 256
    ws = p.alloc("ws", 2 * C * E + C)
    p.add(R.K_TEMPORAL_GRAD_SCAN, [g, rs, out, E, T, ws, 0], [44100.0], label="scan")
    p.output_cell = "out"
    return p


def scan64(g, rs):
    """The same scan in fp64 (the rounding-free value both fp32 scans approximate)."""
    out = np.zeros(g.shape)
    carry = np.zeros(g.shape[1])
    for n in range(g.shape[0] - 1, -1, -1):
        active = 0.0 * carry if rs[n] > 0 else carry
        out[n] = active
        carry = g[n] + active
    return out


@pytest.mark.parametrize("E,T", [(256, (1 << 16) + 123), (1, 5000), (70, 256)])
def test_scan_matches_oracle(gpu, E, T):
    rng = np.random.default_rng(E + T)
    g = rng.standard_normal((T, E)).astype(np.float32)
    n = np.arange(T)
    resets = {"none": np.zeros(T), "every 1000": (n % 1000 == 999), "from half": n >= T // 2,
              "isolated": np.isin(n, [0, 255, 256, T - 1]), "all": np.ones(T)}
    with R.HIPLazyRuntime(scan_program(E, T), 0) as rt:
        rt.write("g", g)
        for name, rs in resets.items():
            rs = np.asarray(rs, np.float32)
            rt.write("reset", rs)
            rt.runNoCopy()
            got = rt.read("out").reshape(T, E)
            ref = O.temporal_scan(g, rs)
            ref64 = scan64(g, rs)
            e_hip, e_o32 = np.abs(got - ref64).max(), np.abs(ref - ref64).max()
            scale = np.abs(ref64).max() + 1.0
            print(f"E={E} T={T} resets {name}: max|out - fp64| HIP {e_hip:.3e}, fp32 oracle {e_o32:.3e} "
                  f"(max |out| {scale - 1:.3e})")
            # the chunked scan reassociates only the carries between chunks:
            # within 2x the sequential fp32 oracle's rounding
            assert e_hip <= 2.0 * e_o32 + 1e-6 * scale
            assert np.all(got[rs > 0] == 0.0)  # a reset frame discards its increment


@pytest.mark.parametrize("E,T", [(1, 4), (3, 31), (64, 32), (65, 67), (70, 68), (256, 131), (5, 132), (130, 1027),
                                 (64, 6 * 32), (2, 4099), (33, 40000)])
@pytest.mark.parametrize("form", ["rising", "resets", "falling", "inf"])
def test_swept_phasor_passes_equal_the_one_pass_loop(E, T, form):
    """With a scratch cell the increments, the phase chain and the loss run as
    separate passes: phase and upstream gradient are the one-pass loop's bit
    for bit over every edge of the 64-frame intervals and segments,
    with resets, negative increments and non-finite ones; the loss, fp64 sums
    in another order rounded to fp32 at the end, to one ulp (1.2e-7)."""
    rng = np.random.default_rng(E * 7 + T)
    slope = rng.uniform(-3e4, 3e4, E) if form == "falling" else rng.uniform(100, 3e4, E)
    time = np.arange(T) / 44100.0
    if form == "inf":
        time[rng.integers(0, T, 2)] = [np.inf, 1e35]
    reset = np.zeros(T) if form in ("rising", "falling") else (rng.random(T) < 0.02).astype(np.float64)
    got = {}
    for scratch in (0, 1):
        p = Program(max_frames=T)
        c = {n: p.alloc(n, k) for n, k in (("slope", E), ("time", T), ("reset", T), ("phase", T * E), ("g", T * E),
                                           ("loss", E), ("scratch", T * E))}
        p.add(R.K_SWEPT_PHASOR, [c["slope"], c["time"], c["reset"], c["phase"], c["g"], c["loss"], E, T, 1,
                                 c["scratch"], scratch], [44100.0, -20.0 if form == "falling" else 80.0, 0.08])
        with R.HIPLazyRuntime(p) as rt:
            for n, a in (("slope", slope), ("time", time), ("reset", reset)):
                rt.write(n, a)
            for _ in range(2):
                rt.runNoCopy()
            got[scratch] = [rt.read(n) for n in ("phase", "g", "loss")]
    for a, b in zip(got[0][:2], got[1][:2]):
        np.testing.assert_array_equal(a, b)
    np.testing.assert_allclose(got[1][2], got[0][2], rtol=1.2e-7)


@pytest.mark.parametrize("shared", ["upstream over the slopes", "loss over the slopes", "phase is upstream",
                                    "scratch is upstream", "scratch is phase"])
def test_swept_phasor_in_place_runs_in_one_pass(gpu, shared):
    """An op with a scratch cell that writes over its inputs, or whose scratch
    is one of its outputs, leaves what the one-pass loop leaves."""
    E, T = 40, 1027
    rng = np.random.default_rng(3)
    slope, time = rng.uniform(100, 3e4, E), np.arange(T) / 44100.0
    got = []
    for scratch in (0, 1):
        p = Program(max_frames=T)
        c = {n: p.alloc(n, k) for n, k in (("time", T), ("reset", T), ("phase", T * E), ("g", T * E), ("loss", E),
                                           ("scratch", T * E), ("slope", E))}
        sl = {"upstream over the slopes": c["g"]}.get(shared, c["slope"])
        lp = sl if shared == "loss over the slopes" else c["loss"]
        ph = c["g"] if shared == "phase is upstream" else c["phase"]
        sc = {"scratch is upstream": c["g"], "scratch is phase": c["phase"]}.get(shared, c["scratch"])
        p.add(R.K_SWEPT_PHASOR, [sl, c["time"], c["reset"], ph, c["g"], lp, E, T, 1, sc, scratch],
              [44100.0, 80.0, 0.08])
        print(f"case {shared}, scratch {scratch}", flush=True)
        with R.HIPLazyRuntime(p) as rt:
            for n, a in (("slope", slope), ("time", time)):
                rt.write(n, a)
            if sl == c["g"]:
                rt.write("g", np.concatenate([slope, np.zeros(T * E - E)]))
            rt.runNoCopy()
            got.append([rt.read(n) for n in ("phase", "g", "loss", "slope")])
    assert np.abs(got[0][1]).max() > 0
    for a, b in zip(*got):
        np.testing.assert_array_equal(a, b)


@pytest.mark.parametrize("reset_from", [-1, 40000])
def test_swept_phasor_gradient(gpu, reset_from):
    cfg = SweptPhasorConfig(reset_from=reset_from)
    print(f"swept phasor bank E={cfg.E} T={cfg.T} reset_from={reset_from}", flush=True)
    s = SweptPhasorSession(cfg, optimizer=False)
    try:
        s.step()
        loss, g = s.loss(), s.rt.read("grads").astype(np.float64)
    finally:
        s.close()
    slopes = cfg.slopes()
    args = (cfg.T, cfg.sr, cfg.base, cfg.target, reset_from, cfg.smooth)
    l64, g64, _ = O.swept_phasor_step(slopes.astype(np.float64), *args)
    l32, g32, _ = O.swept_phasor_step(slopes, *args, prec="f32")
    e_hip, e_o32 = np.linalg.norm(g - g64) / np.linalg.norm(g64), np.linalg.norm(g32 - g64) / np.linalg.norm(g64)
    print(f"loss {loss:.6e} (fp64 oracle {l64:.6e}); grad rel L2 vs fp64: HIP {e_hip:.3e}, fp32 oracle {e_o32:.3e}")
    assert abs(loss - l64) <= 1e-4 * abs(l64)
    assert e_hip <= 2.0 * e_o32 + 1e-5
    for e in (0, cfg.E // 2, cfg.E - 1):  # central differences of the fp64 oracle, one lane at a time
        sl = np.array([slopes[e]], np.float64)
        eps = 1e-7 * sl[0]
        lp = O.swept_phasor_step(sl + eps, *args, grad=False)[0]
        lm = O.swept_phasor_step(sl - eps, *args, grad=False)[0]
        d = (lp - lm) / (2 * eps)
        print(f"lane {e} slope {sl[0]:.1f}: HIP {g[e]:.6e}, FD {d:.6e}")
        # fp32 phases: lanes whose gradient cancels to a few units carry the
        # bank's absolute fp32 error, hence the floor at 1e-3 of the largest
        assert abs(g[e] - d) <= 1e-2 * abs(d) + 1e-3 * np.abs(g64).max()
