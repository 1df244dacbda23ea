"""Performance cases: the workloads a program runs through this framework's
public entry points (schedule builders, sessions, ``HIPLazyRuntime``), over
the range of sizes its configurations, tests and benchmark use.

A training pass is one step of a training loop (forward, loss, backward,
optimiser) followed by what the loop looks at: the loss, the gradients and,
where they are few, the updated parameters, read through the runtime's host
memory.  A render pass returns the audio.  A streaming pass is one process
call on host channel buffers.
"""
from __future__ import annotations

import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "dgen-audio_amd"))
import dgen_hip.programs as P  # noqa: E402
from dgen_hip import (BiquadConfig, HarmonicConfig, HIPLazyRuntime, MembraneConfig, OscBankConfig,  # noqa: E402
                      StftConfig, SvfConfig, SweptPhasorConfig)
from dgen_hip.programs import HarmonicSession  # noqa: E402

FFT_SETS = {"six": (2048, 1024, 512, 256, 128, 64), "two": (512, 256), "three": (1024, 256, 64)}
F64 = torch.float64


def listed():
    return [
        # one short signal: an oscillator bank through a one-pole, rendered whole
        dict(name="osc_bank", kind="osc", n_osc=16, frames=65536, graphs=False),
        # a host's audio callback: one block of a stateful filter bank on host buffers
        dict(name="stream_biquad_block", kind="stream", B=16, frames=512),
        # a render-only spectral filter of two short clips, odd length
        dict(name="stft_render", kind="stft", S=2, T=44101, N=512, H=128, train=False, graphs=False),
        # learning a spectral filter on eight long signals
        dict(name="stft_train", kind="stft", S=8, T=1 << 20, N=1024, H=256, train=True, graphs=True),
        # a voice's filter fitted over one short note, a dozen candidates at once
        dict(name="biquad_train_voice", kind="biquad", B=12, T=8192, graphs=False),
        # the filter bank over long signals
        dict(name="biquad_train_bank", kind="biquad", B=256, T=1 << 18, graphs=True),
        # the linear state-variable filter with a cutoff envelope, odd sizes
        dict(name="svf_train_linear", kind="svf", B=70, T=30001, saturating=False, graphs=False),
        # the saturating state-variable filter with a learnable drive per lane
        dict(name="svf_train_saturating", kind="svf", B=256, T=1 << 16, saturating=True, graphs=True),
        # learning sweep rates through the phase accumulator's temporal gradient
        dict(name="swept_phasor_train", kind="sweep", E=256, T=1 << 16, smooth=True, reset_from=-1, graphs=True),
        # the 2D membrane fitted to a recorded pickup
        dict(name="membrane_train", kind="membrane", R=512, C=512, T=1200, graphs=True),
        # a small harmonic model trained on short clips, odd sizes, two FFT sizes
        dict(name="harmonic_train_small", kind="harmonic", B=3, T=8003, K=24, NF=33, hidden=96, fft="two", train=True,
             graphs=False),
        # the batch-32 harmonic synth's training step, as the benchmark runs it
        dict(name="harmonic_train_b32", kind="harmonic", B=32, T=64000, K=60, NF=65, hidden=512, fft="six", train=True,
             graphs=True),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["osc", "stream", "stft", "biquad", "svf", "svf", "sweep", "membrane", "harmonic", "harmonic"])
    graphs = rng.random() < 0.5
    if kind == "osc":
        return dict(kind=kind, n_osc=_log(rng, 1, 64), frames=_log(rng, 64, 1 << 18), graphs=graphs)
    if kind == "stream":
        return dict(kind=kind, B=_log(rng, 1, 64), frames=_log(rng, 32, 2048))
    if kind == "stft":
        N = rng.choice([64, 128, 256, 512, 1024, 2048])
        return dict(kind=kind, S=rng.randint(1, 8), T=_log(rng, 4096, 1 << 20), N=N, H=N // rng.choice([1, 2, 4, 4]),
                    train=rng.random() < 0.7, graphs=graphs)
    if kind == "biquad":
        return dict(kind=kind, B=_log(rng, 4, 256), T=_log(rng, 2048, 1 << 18), graphs=graphs)
    if kind == "svf":
        return dict(kind=kind, B=_log(rng, 4, 256), T=_log(rng, 2048, 1 << 16), saturating=rng.random() < 0.5,
                    graphs=graphs)
    if kind == "sweep":
        T = _log(rng, 1024, 1 << 16)
        return dict(kind=kind, E=_log(rng, 1, 256), T=T, smooth=rng.random() < 0.7,
                    reset_from=rng.choice([-1, T // 2]), graphs=graphs)
    if kind == "membrane":
        return dict(kind=kind, R=_log(rng, 32, 512), C=_log(rng, 32, 512), T=_log(rng, 64, 1200), graphs=graphs)
    return dict(kind=kind, B=_log(rng, 1, 32), T=_log(rng, 2048, 32000), K=rng.randint(8, 100), NF=rng.randint(9, 100),
                hidden=rng.choice([64, 96, 128, 256, 384, 512]), fft=rng.choice(sorted(FFT_SETS)),
                train=rng.random() < 0.7, graphs=graphs)


# ------------------------------------------------------------------ inputs
def _rng(case, seed):
    return np.random.default_rng([int(seed) & 0xFFFFFFFF, sum(map(ord, case["kind"]))])


def _config(case):
    k = case["kind"]
    if k == "osc":
        return OscBankConfig(n_osc=case["n_osc"], frames=case["frames"])
    if k == "stream":
        return BiquadConfig(B=case["B"], T=case["frames"])
    if k == "stft":
        return StftConfig(S=case["S"], T=case["T"], N=case["N"], H=case["H"])
    if k == "biquad":
        return BiquadConfig(B=case["B"], T=case["T"])
    if k == "svf":
        return SvfConfig(B=case["B"], T=case["T"], saturating=case["saturating"])
    if k == "sweep":
        return SweptPhasorConfig(E=case["E"], T=case["T"], smooth=case["smooth"], reset_from=case["reset_from"])
    if k == "membrane":
        return MembraneConfig(R=case["R"], C=case["C"], T=case["T"])
    return HarmonicConfig(B=case["B"], T=case["T"], K=case["K"], NF=case["NF"], hidden=case["hidden"],
                          fft_sizes=FFT_SETS[case["fft"]])


def _noise(r, shape):
    """U[-1, 1) in fp32."""
    a = r.random(shape, dtype=np.float32)
    a *= 2.0
    a -= 1.0
    return a


def _inputs(case, seed):
    """The cells a program writes, by name."""
    r, cfg, k = _rng(case, seed), _config(case), case["kind"]
    if k == "osc":
        amps = r.random(cfg.n_osc)
        return dict(freqs=(np.arange(1, cfg.n_osc + 1) * r.uniform(55.0, 330.0)).astype(np.float32),
                    amps=(amps / amps.sum()).astype(np.float32))
    if k in ("stream", "biquad"):
        prm = np.concatenate([r.uniform(120.0, 400.0, cfg.B), r.uniform(0.5, 2.0, cfg.B)]).astype(np.float32)
        d = dict(x=_noise(r, (cfg.T, cfg.B)), mod=cfg.modulation(), params=prm)
        if k == "biquad":
            d["target"] = _noise(r, (cfg.T, cfg.B))
        return d
    if k == "stft":
        x = r.standard_normal((cfg.S, cfg.T), dtype=np.float32)
        x *= cfg.sigma
        return dict(x=x, window=cfg.window(), gains=r.uniform(0.4, 1.2, cfg.bins).astype(np.float32))
    if k == "svf":
        u = r.random((3, cfg.B))
        rows = [cfg.base_lo * (cfg.base_hi / cfg.base_lo) ** u[0], cfg.res_lo + (cfg.res_hi - cfg.res_lo) * u[1]]
        rows += [cfg.ks_hi * u[2]] if cfg.saturating else []
        return dict(x=_noise(r, (cfg.T, cfg.B)), target=_noise(r, (cfg.T, cfg.B)), mod=cfg.modulation(),
                    env=cfg.envelope(), params=np.concatenate(rows).astype(np.float32))
    if k == "sweep":
        s = cfg.slope_lo * (cfg.slope_hi / cfg.slope_lo) ** r.random(cfg.E)
        return dict(slope=s.astype(np.float32), reset=cfg.reset())
    if k == "membrane":
        u0 = MembraneConfig(R=cfg.R, C=cfg.C, T=cfg.T, seed=int(r.integers(1, 1 << 30))).bump()
        n = np.arange(cfg.T)
        tgt = 0.05 * np.exp(-n / 600.0) * np.sin(n * r.uniform(0.02, 0.2))
        return dict(u0=u0, target=tgt.astype(np.float32), params=cfg.params())
    # f0 tracks (a random walk per lane), loudness, an init of the trainer's
    # scale, and as the target a quiet harmonic recording of other pitches
    B, F, T = cfg.B, cfg.F, cfg.T
    walk = np.cumsum(r.standard_normal((F, B)) * 0.01, axis=0)
    f0 = np.exp(r.uniform(math.log(60.0), math.log(900.0), B)[None, :] + walk - walk[:1]).astype(np.float32)
    lo, hi = math.log(cfg.min_f0), math.log(cfg.max_f0)
    X = np.empty((B * F, cfg.din), np.float32)
    X[:, 0] = ((np.log(np.maximum(f0, cfg.min_f0)) - lo) / (hi - lo)).T.reshape(-1)
    X[:, 1] = r.random(B * F)
    parts, fan = [], cfg.din
    for _ in range(cfg.layers):
        parts += [_noise(r, fan * cfg.hidden) * np.float32(math.sqrt(2.0 / fan) * 0.5), np.zeros(cfg.hidden, np.float32)]
        fan = cfg.hidden
    bh = np.zeros(cfg.NC, np.float32)
    bh[cfg.K + 1] = -3.0
    parts += [_noise(r, cfg.hidden * cfg.NC) * np.float32(0.05), bh]
    d = dict(f0=f0, uv=np.ones((F, B), np.float32), X=X, params=np.concatenate(parts))
    if case["train"]:
        t = np.arange(T, dtype=np.float32)[None, :] * np.float32(2.0 * math.pi / cfg.sr)
        w = r.uniform(80.0, 700.0, (B, 1)).astype(np.float32)
        d["target"] = (0.2 * np.sin(t * w) + 0.1 * np.sin(t * (w * 2)) + 0.01 * _noise(r, (B, T))).astype(np.float32)
    return d


class _Held(np.ndarray):
    """A view of a runtime's host memory that keeps the runtime open."""


def _view(rt, a):
    v = a.view(_Held)
    v.rt = rt
    return v


def _cell(rt, name):
    rt.download(name)
    c = rt.program.cells[name]
    return _view(rt, rt.memoryPointer()[c.off:c.off + c.n])


TRAIN_CELLS = {"stft": ("loss", "grads", "gains"), "biquad": ("loss", "grads", "params"),
               "svf": ("loss", "grads", "params"), "sweep": ("loss", "grads", "slope"),
               "membrane": ("loss", "grads", "params"), "harmonic": ("loss_frames", "grads")}


def prepare(case, seed):
    cfg, k, d = _config(case), case["kind"], _inputs(case, seed)
    train = case.get("train", k not in ("osc", "stream"))
    s = dict(kind=k, train=train)
    if k == "harmonic" and train:
        sess = HarmonicSession(cfg, target=d["target"], data=(d["f0"], d["uv"], d["X"]))
        sess.rt.write("params", d["params"])
        s.update(sess=sess, rt=sess.rt)
    else:
        if k == "osc":
            prog = P.oscbank_program(cfg)
        elif k == "stream":
            prog = P.stream_biquad_program(cfg)
        elif k == "stft":
            prog = P.stft_program(cfg, train=train)
        elif k == "biquad":
            prog = P.biquad_program(cfg)
        elif k == "svf":
            prog = P.svf_program(cfg)
        elif k == "sweep":
            prog = P.swept_phasor_program(cfg)
        elif k == "membrane":
            prog = P.membrane_program(cfg)
        else:
            prog = P.harmonic_program(cfg, train=False)
        rt = s["rt"] = HIPLazyRuntime(prog)
        if k == "stream":
            rt.write("params", d["params"])
            rt.setProcessPorts(*prog.meta["ports"])
            s["ins"] = [np.ascontiguousarray(d["x"][:, b]) for b in range(cfg.B)] + [d["mod"]]
            s["frames"] = cfg.T
        else:
            for name, a in d.items():
                rt.write(name, a)
    if train:
        s["rt"].setOutputs(None)  # a training loop does not fetch the audio of every step
        s["cells"] = TRAIN_CELLS[k]
    if case.get("graphs"):
        s["rt"].set_graphs(True)
    return s


def run(state):
    rt = state["rt"]
    if state["kind"] == "stream":
        return rt.process(state["ins"], state["frames"])
    if not state["train"]:
        rt.runNoCopy()
        return _view(rt, rt.outputsPointer())
    if "sess" in state:
        state["sess"].step()
    else:
        rt.runNoCopy()
    return {name: _cell(rt, name) for name in state["cells"]}


# -------------------------------------------------------------------- work
def work(case):
    cfg, k = _config(case), case["kind"]
    if k == "osc":
        return dict(bytes=8.0 * cfg.n_osc + 4.0 * cfg.frames, flops=cfg.frames * (26.0 * cfg.n_osc + 2.0))
    if k == "stream":
        return dict(bytes=8.0 * cfg.T * cfg.B + 4.0 * cfg.T, flops=25.0 * cfg.T * cfg.B)
    if k == "stft":
        n, nwin = float(cfg.S * cfg.T), cfg.S * ((cfg.T + cfg.H - 1) // cfg.H)
        fft = 2.5 * cfg.N * math.log2(cfg.N)
        if not case["train"]:
            return dict(bytes=8.0 * n, flops=nwin * 2 * fft)
        return dict(bytes=4.0 * n + 28.0 * cfg.bins, flops=nwin * (3 * fft + 4 * cfg.bins))
    if k in ("biquad", "svf"):
        n = float(cfg.T * cfg.B)
        per = 70.0 if k == "biquad" else 110.0
        return dict(bytes=8.0 * n + 4.0 * cfg.T, flops=per * n)
    if k == "sweep":
        return dict(bytes=28.0 * cfg.E + 4.0 * cfg.T, flops=14.0 * cfg.E * cfg.T)
    if k == "membrane":
        return dict(bytes=4.0 * cfg.R * cfg.C + 8.0 * cfg.T, flops=24.0 * cfg.R * cfg.C * cfg.T)
    M, H, n = cfg.M, cfg.hidden, float(cfg.B * cfg.T)
    mlp = 2.0 * M * (cfg.din * H + (cfg.layers - 1) * H * H + H * cfg.NC)
    synth = n * (35.0 * cfg.K + 5.0 * cfg.NF)
    data = 4.0 * (M * cfg.din + 2 * M + cfg.param_count())
    if not case["train"]:
        return dict(bytes=data + 4.0 * n, flops=mlp + synth)
    fft = sum(((cfg.T + N // 4 - 1) // (N // 4)) * cfg.B * (7.5 * N * math.log2(N) + 30.0 * N) for N in cfg.fft_sizes)
    return dict(bytes=data + 4.0 * n + 4.0 * cfg.T + 24.0 * cfg.param_count(),
                flops=3.0 * mlp + 2.0 * synth + n * (6.0 * cfg.K + 4.0 * cfg.NC) + fft)


def tolerance(case):
    k = case["kind"]
    if k == "harmonic":
        # the log-magnitude loss divides by the magnitude of near-silent bins,
        # so fp32 rounding anywhere before it moves the whole gradient by
        # percents; the audio itself is well conditioned
        return {"rel": 0.03, "max": 0.99} if case["train"] else {"rel": 5e-6}
    # about four times the distance from the 64-bit result, which the lowest
    # cutoffs set for the filters' audio, the fp32 phase's rounding for the
    # sweep and the near-cancelling Laplacian for the membrane's gradient
    return {"rel": {"osc": 5e-6, "stream": 1e-5, "stft": 5e-6, "biquad": 1e-5, "svf": 1e-5, "sweep": 3e-5,
                    "membrane": 3e-4}[k]}


# ------------------------------------------------- the same in 64 bits
DEV = "cuda" if torch.cuda.is_available() else "cpu"


def _t(a):
    return torch.as_tensor(np.ascontiguousarray(a), device=DEV).to(F64)


def _adam(p, g, lr):
    """The first Adam step from zero moments."""
    return p - lr * g / (g.abs() + 1e-8)


def _affine_scan(A, b):
    """States entering every step of s' = A[n] s + b[n], s = 0 before step 0:
    A [T,B,2,2], b [T,B,2] -> [T,B,2].  Chunks run side by side from the zero
    state and the two unit states, then are joined in order."""
    T, B = b.shape[:2]
    L = max(1, int(math.sqrt(T)))
    C = (T + L - 1) // L
    pad = C * L - T
    A = torch.cat([A, A.new_zeros(pad, B, 2, 2)]).view(C, L, B, 2, 2)
    b = torch.cat([b, b.new_zeros(pad, B, 2)]).view(C, L, B, 2)
    zs, M = b.new_empty(C, L + 1, B, 2), A.new_empty(C, L + 1, B, 2, 2)
    zs[:, 0] = 0
    M[:, 0] = torch.eye(2, dtype=F64, device=A.device)
    for i in range(L):
        zs[:, i + 1] = (A[:, i] * zs[:, i, :, None, :]).sum(-1) + b[:, i]
        M[:, i + 1] = (A[:, i, :, :, :, None] * M[:, i, :, None, :, :]).sum(-2)
    s, out = b.new_zeros(B, 2), b.new_empty(C, L, B, 2)
    for c in range(C):
        out[c] = zs[c, :L] + (M[c, :L] * s[None, :, None, :]).sum(-1)
        s = zs[c, L] + (M[c, L] * s[:, None, :]).sum(-1)
    return out.view(C * L, B, 2)[:T]


def _jacobian(step, S, prm):
    """Per-frame derivatives of (s1', s2', y) by (s1, s2): [T,B,3,2]."""
    s = S.detach().requires_grad_(True)
    outs = step(s[..., 0], s[..., 1], prm)
    return torch.stack([torch.autograd.grad(o.sum(), s, retain_graph=True)[0] for o in outs], -2)


def _bptt(step, S, prm, tgt):
    """Loss sum (y - tgt)^2 and its gradient by the parameters, from the
    states S entering every frame of the recurrence `step`."""
    J = _jacobian(step, S, prm)
    p = prm.detach().requires_grad_(True)
    n1, n2, y = step(S[..., 0], S[..., 1], p)
    e = 2.0 * (y.detach() - tgt)
    # the adjoint entering frame n from its end: l_n = J_n^T l_{n+1} + C_n e_n
    back = _affine_scan(J[..., :2, :].transpose(-1, -2).flip(0), (J[..., 2, :] * e[..., None]).flip(0)).flip(0)
    g, = torch.autograd.grad((back[..., 0] * n1 + back[..., 1] * n2 + e * y).sum(), p)
    return ((y.detach() - tgt) ** 2).sum(), g


def _biquad_step(d, T, B):
    x, m = _t(d["x"]), _t(d["mod"])[:, None]
    z = x.new_zeros(1, B)
    x1, x2 = torch.cat([z, x])[:T], torch.cat([z, z, x])[:T]

    def step(y1, y2, prm):
        w = (prm[:B] * m).abs() * float(np.float32(0.00014247585730565955))
        q, c, s = prm[B:].abs(), torch.cos(w), torch.sin(w)
        alpha = s * 0.5 / q
        r = 1.0 / (alpha + 1.0)
        b1 = (1.0 - c) * r
        y = b1 * (0.5 * x + x1 + 0.5 * x2) - ((1.0 - alpha) * r * y2 - 2.0 * c * r * y1)
        return y, y1 + 0.0 * y, y
    return step


def _svf_coefs(d, B, prm, sr):
    raw = prm[:B] * _t(d["mod"])[:, None] + _t(d["env"])[:, None]
    g = torch.tan(float(np.float32(math.pi)) * torch.clamp(raw, 20.0, 20000.0) / sr)
    a1 = 1.0 / (1.0 + g * (g + 1.0 / prm[B:2 * B]))
    return g, a1, g * a1


def _svf_step(d, B, sr, sat):
    x = _t(d["x"])

    def step(c1, c2, prm):
        g, a1, a2 = _svf_coefs(d, B, prm, sr)
        s1, s2 = (c / (1.0 + (prm[2 * B:] * c).abs()) for c in (c1, c2)) if sat else (c1, c2)
        v1 = a1 * s1 + a2 * (x - s2)
        i1 = 2.0 * v1 - s1
        i2 = 2.0 * (s2 + g * ((i1 + s1) * 0.5)) - s2
        return i1, i2, (i2 + s2) * 0.5
    return step


def _exact_filter(case, cfg, d):
    T, B, sat = cfg.T, cfg.B, case.get("saturating", False)
    prm, biquad = _t(d["params"]), case["kind"] != "svf"
    step = _biquad_step(d, T, B) if biquad else _svf_step(d, B, cfg.sr, sat)
    if sat:
        g, a1, a2 = (v.cpu().numpy() for v in _svf_coefs(d, B, prm, cfg.sr))
        x, ks = d["x"].astype(np.float64), d["params"][2 * B:].astype(np.float64)
        S, c1, c2 = np.empty((T, B, 2)), np.zeros(B), np.zeros(B)
        for n in range(T):
            S[n, :, 0], S[n, :, 1] = c1, c2
            s1, s2 = c1 / (1.0 + np.abs(ks * c1)), c2 / (1.0 + np.abs(ks * c2))
            c1 = 2.0 * (a1[n] * s1 + a2[n] * (x[n] - s2)) - s1
            c2 = 2.0 * (s2 + g[n] * ((c1 + s1) * 0.5)) - s2
        S = torch.as_tensor(S, device=DEV)
    else:
        zero = torch.zeros(T, B, 2, dtype=F64, device=DEV)
        b = torch.stack(step(zero[..., 0], zero[..., 1], prm)[:2], -1)
        S = _affine_scan(_jacobian(step, zero, prm)[..., :2, :], b)
    if case["kind"] == "stream":
        return step(S[..., 0], S[..., 1], prm)[2].T.contiguous()
    loss, g = _bptt(step, S, prm, _t(d["target"]))
    return dict(loss=loss.reshape(1), grads=g, params=_adam(prm, g, cfg.lr))


def _exact_osc(cfg, d):
    # the phase is the graph's fp32 expression; everything after it in 64 bits
    inc = d["freqs"] / np.float32(cfg.sr)
    r = inc[None, :] * np.arange(cfg.frames, dtype=np.float32)[:, None]
    ph = (r - np.floor(r)).astype(np.float64)
    x = (np.sin(ph * float(np.float32(2.0 * math.pi))) * d["amps"].astype(np.float64)).sum(1)
    y, pole = 0.0, float(np.float32(cfg.pole))
    out = np.empty(cfg.frames)
    for n, v in enumerate(x.tolist()):
        y = v + pole * y
        out[n] = y
    return out


def _exact_stft(case, cfg, d):
    S, T, N, H = cfg.S, cfg.T, cfg.N, cfg.H
    x, win, g = _t(d["x"]), _t(d["window"]), _t(d["gains"])
    nwin = (T + H - 1) // H
    xp = torch.cat([x.new_zeros(S, N - 1), x, x.new_zeros(S, N)], 1)
    spec = torch.fft.rfft(xp.unfold(1, N, H)[:, :nwin] * win)
    z = torch.fft.irfft(spec * g, n=N)
    y = torch.nn.functional.fold(z.transpose(1, 2), (1, (nwin - 1) * H + N), (1, N), stride=(1, H))[:, 0, 0, :T]
    if not case["train"]:
        return y.reshape(-1)
    dy = 2.0 * (y - x) / T
    e = torch.fft.rfft(torch.cat([dy, dy.new_zeros(S, N + H)], 1).unfold(1, N, H)[:, :nwin])
    c = torch.full((cfg.bins,), 2.0 / N, dtype=F64, device=DEV)
    c[0] = c[-1] = 1.0 / N
    dg = (spec.real * e.real + spec.imag * e.imag).sum((0, 1)) * c
    return dict(loss=((y - x) ** 2).sum().reshape(1) / T, grads=dg, gains=_adam(g, dg, cfg.lr))


def _accum(T, step, span):
    """The fp32 accumulator from 0, wrapping at `span`: values before each update."""
    out, st, step, span = np.empty(T, np.float32), np.float32(0), np.float32(step), np.float32(span)
    for n in range(T):
        out[n] = st
        w = st + step
        w = w - np.floor(w / span) * span
        st = w - span if w >= span else w
    return out


def _phases(inc, reset=None):
    """The fp32 phase before each frame's update: inc [T, lanes]."""
    out, ph = np.empty_like(inc), np.zeros(inc.shape[1], np.float32)
    for n in range(inc.shape[0]):
        out[n] = ph
        ph = ph + inc[n]
        ph -= np.floor(ph)
        ph[ph >= 1.0] -= np.float32(1.0)
        if reset is not None and reset[n] > 0:
            ph[:] = 0.0
    return out


def _exact_sweep(cfg, d):
    sr, two_pi = np.float32(cfg.sr), float(np.float32(2.0 * math.pi))
    time = _accum(cfg.T, np.float32(1.0) / sr, 1.0)
    inc = (np.float32(cfg.base) + d["slope"][None, :] * time[:, None]) / sr
    ph, rs = _t(_phases(inc, d["reset"])), _t(d["reset"])
    v = torch.sin(ph * two_pi) if cfg.smooth else ph
    e = v - float(np.float32(cfg.target))
    up = 2.0 * e * (torch.cos(ph * two_pi) * two_pi if cfg.smooth else 1.0)
    # the gradient reaching frame n's increment: the upstream of the later
    # frames, up to and with the next reset frame (none from a reset frame itself)
    incl = up.flip(0).cumsum(0).flip(0)
    suf = incl - up
    if (rs > 0).any():
        n0 = int((rs > 0).nonzero()[0, 0])
        suf = suf - (incl[n0 + 1:n0 + 2] if n0 + 1 < cfg.T else 0.0)
        suf[n0:] = 0.0
    g = (suf / float(sr) * _t(time)[:, None]).sum(0)
    return dict(loss=(e * e).sum().reshape(1), grads=g, slope=_adam(_t(d["slope"]), g, cfg.lr))


def _exact_membrane(cfg, d):
    R, C, T = cfg.R, cfg.C, cfg.T
    prm, tgt = _t(d["params"]), _t(d["target"])
    c2, dd = float(prm[0]), float(prm[1])
    py, px = cfg.pickup

    def lap(u):
        o = -4.0 * u
        o[1:] += u[:-1]
        o[:-1] += u[1:]
        o[:, 1:] += u[:, :-1]
        o[:, :-1] += u[:, 1:]
        return o
    U = torch.empty(T + 2, R, C, dtype=F64, device=DEV)
    U[0] = U[1] = _t(d["u0"]).reshape(R, C)
    for n in range(T):
        U[n + 2] = 2.0 * U[n + 1] - U[n] + c2 * lap(U[n + 1]) - dd * (U[n + 1] - U[n])
    e = U[2:, py, px] - tgt
    l1, l2, gc, gd = torch.zeros_like(U[0]), torch.zeros_like(U[0]), 0.0, 0.0
    for n in range(T, 0, -1):
        lam = (2.0 - dd) * l1 + c2 * lap(l1) - (1.0 - dd) * l2
        lam[py, px] += 2.0 * e[n - 1]
        gc = gc + (lam * lap(U[n])).sum()
        gd = gd + (lam * (U[n - 1] - U[n])).sum()
        l1, l2 = lam, l1
    g = torch.stack([gc, gd])
    return dict(loss=(e * e).sum().reshape(1), grads=g, params=_adam(prm, g, cfg.lr))


def _exact_harmonic(case, cfg, d):
    B, F, T, K, NF, NC, Hd = cfg.B, cfg.F, cfg.T, cfg.K, cfg.NF, cfg.NC, cfg.hidden
    f32 = np.float32
    # the data path is the graph's fp32 program: playhead, row weights, f0
    # frames, the phase accumulators and the noise
    top = f32(max(0, F - 1))
    play = np.clip(_accum(T, top / f32(max(1, T - 1)), top if F > 1 else 1.0), f32(0), max(f32(0), top - f32(1e-4)))
    fl = np.floor(play)
    lo, hi = fl.astype(np.int64), (fl.astype(np.int64) + 1) % F
    frac = (play - fl).astype(f32)
    omf = f32(1.0) - frac
    f0 = omf[:, None] * d["f0"][lo] + frac[:, None] * d["f0"][hi]  # [T][B]
    freq = f0[:, :, None] * np.arange(1, K + 1, dtype=f32)
    phase = _phases((freq / f32(cfg.sr)).reshape(T, B * K)).reshape(T, B, K)
    mask = freq < f32(cfg.sr * 0.5)
    noise, s = np.empty(T), 1
    for t in range(T):
        s ^= (s << 13) & 0xFFFFFFFF
        s ^= s >> 17
        s ^= (s << 5) & 0xFFFFFFFF
        noise[t] = float(f32(s)) / 4294967296.0
    lo, hi, frac, omf = (torch.as_tensor(v, device=DEV) for v in (lo, hi, _t(frac), _t(omf)))
    taps = torch.cat([torch.zeros(NF - 1, dtype=F64, device=DEV), _t(noise)]).unfold(0, NF, 1)
    # control network
    prm = _t(d["params"]).requires_grad_(True)
    h, off, fan = _t(d["X"]), 0, cfg.din
    for _ in range(cfg.layers):
        W, b = prm[off:off + fan * Hd].view(fan, Hd), prm[off + fan * Hd:off + fan * Hd + Hd]
        h, off, fan = torch.tanh(h @ W + b), off + fan * Hd + Hd, Hd
    z = h @ prm[off:off + Hd * NC].view(Hd, NC) + prm[off + Hd * NC:]
    amp = torch.nn.functional.softplus(z[:, :K + 2], threshold=700.0)
    fir = torch.tanh(z[:, K + 2:])
    ctrl = torch.cat([amp[:, :K] / (amp[:, :K].sum(1, keepdim=True) + 1e-6), amp[:, K:],
                      fir / (fir.abs().sum(1, keepdim=True) + 1e-4)], 1).view(B, F, NC)
    leaf = ctrl.detach().requires_grad_(True)
    hann = {N: 0.5 * (1.0 - torch.cos(2.0 * math.pi * torch.arange(N, dtype=F64, device=DEV) / (N - 1)))
            for N in cfg.fft_sizes}
    frames, ys = torch.zeros(T, dtype=F64, device=DEV), []
    wl, wg = cfg.w_lin / len(cfg.fft_sizes), cfg.w_log / len(cfg.fft_sizes)
    for b in range(B):
        rows = omf[:, None] * leaf[b][lo] + frac[:, None] * leaf[b][hi]
        m = rows[:, :K] * torch.as_tensor(mask[:, b], device=DEV)
        sines = torch.sin(_t(phase[:, b]) * float(f32(2.0 * math.pi)))
        y = ((sines * m).sum(1) / (m.sum(1) + 1e-8) * rows[:, K]
             + (taps * rows[:, K + 2:]).sum(1) * rows[:, K + 1] * float(f32(0.12)))
        if not case["train"]:
            ys.append(y.detach())
            continue
        total = 0.0
        for N in cfg.fft_sizes:
            nw = (T + N // 4 - 1) // (N // 4)

            def mag(v):
                w = torch.cat([v.new_zeros(N - 1), v, v.new_zeros(N)]).unfold(0, N, N // 4)[:nw]
                q = torch.fft.rfft(w * hann[N])
                return torch.sqrt((q.real ** 2 + q.imag ** 2).clamp_min(1e-60))
            m1, m2 = mag(y), mag(_t(d["target"][b]))
            win = (wl * (m1 - m2).abs().sum(1) + wg * (torch.log(m1 + 1e-8) - torch.log(m2 + 1e-8)).abs().sum(1)) / B / T
            frames[::N // 4] += win.detach()
            total = total + win.sum()
        total.backward()
    if not case["train"]:
        return torch.stack(ys).reshape(-1)
    g, = torch.autograd.grad(ctrl, prm, leaf.grad)
    return dict(loss_frames=frames, grads=g)


def exact(case, seed):
    cfg, d, k = _config(case), _inputs(case, seed), case["kind"]
    if k == "osc":
        return _exact_osc(cfg, d)
    if k == "stft":
        return _exact_stft(case, cfg, d)
    if k == "sweep":
        return _exact_sweep(cfg, d)
    if k == "membrane":
        return _exact_membrane(cfg, d)
    if k == "harmonic":
        return _exact_harmonic(case, cfg, d)
    return _exact_filter(case, cfg, d)
