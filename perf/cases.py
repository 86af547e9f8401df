"""Performance cases of the radar signal-processing path, through its public
Python entry points: the two fft_conv sizes of small calls, the pipelines of
`matx_amd.radar`, the ragged batch, the two differentiable objectives, and the
single operators (long-signal convolution, transforms, CFAR, an elementwise
threshold).  Sizes are the ones of the benchmark and of the tests, with odd
and small relatives; `draw` spreads over the same ranges.
"""
from __future__ import annotations

import math

import torch

import matx_amd as mx
from matx_amd import autograd as ag
from matx_amd import expr as E
from matx_amd import ops

DEV = "cuda"


# ------------------------------------------------------------------- cases
def listed():
    return [
        # One small receiver dwell: a handful of kilobyte-sized pulses, where
        # the launch and the call itself are the cost.
        dict(name="fft_conv_1x8x1000", kind="fft_conv", C=1, P=8, S=1000, L=100, n=1024),
        # Plain pulse compression of a short cube, full circular output.
        dict(name="fft_conv_4x32x2048", kind="fft_conv", C=4, P=32, S=2048, L=256, n=4096),
        # The headline radar chain: one cube from raw samples to detections,
        # the waveform prepared once.
        dict(name="radar_16x128x9000", kind="radar", C=16, P=128, S=9000, L=1000, gx=5),
        # The stage-by-stage pipeline on a small cube of odd sizes, new data
        # and a fresh waveform in every pass, power and averages kept.
        dict(name="stages_5x77x5003", kind="stages", C=5, P=77, S=5003, L=487),
        # Waveform design over a whole large cube: forward and backward of
        # 512 pulses of 32768 samples, a quarter of the largest cube's channels.
        dict(name="radar_grad_16x512x32768", kind="radar_grad", C=16, P=512, S=32768, L=4096),
        # Phase-coded waveform and Doppler window design: one gradient step.
        dict(name="design_64x1024", kind="design", B=64, L=1024, n=8192, C=16, P=128, R=4096, T=24),
        # Sixty dwells of uneven shapes as one batch.
        dict(name="ragged_60", kind="ragged", jobs=60, shapes=11),
        # Long recordings through a 209-tap filter by the FFT method.
        dict(name="conv1d_16x1048576", kind="conv1d", rows=16, N=1048576, L=209, mode="same"),
        # A batch of transforms whose length is not a power of two.
        dict(name="fft_8192x1000", kind="fft", a=1, rows=8192, n=1000, cols=1, op="fft"),
        # Doppler transforms of a compressed cube along its strided axis.
        dict(name="fft_16x256x8001_axis1", kind="fft", a=16, rows=0, n=256, cols=8001, op="fft"),
        # Detection alone on a large power map with the wide window.
        dict(name="cfar_8x512x28673", kind="cfar", C=8, Ny=512, Nx=28673, wy=7, wx=21, gy=3, gx=5,
             want_ba=False),
        # The detection threshold as a user's elementwise expression.
        dict(name="expr_16x128x8001", kind="expr", C=16, P=128, R=8001),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["fft_conv", "radar", "radar", "stages", "radar_grad", "design", "ragged",
                       "conv1d", "fft", "fft", "cfar", "expr"])
    if kind == "fft_conv":
        S = _log(rng, 600, 8192)
        n = _pow2(S) * rng.choice([1, 1, 2])
        return dict(kind=kind, C=rng.randint(1, 8), P=_log(rng, 1, 64), S=S,
                    L=_log(rng, 16, S // 4), n=n)
    if kind in ("radar", "stages"):
        S = _log(rng, 1000, 9000)
        c = dict(kind=kind, C=rng.randint(1, 16 if kind == "radar" else 8),
                 P=rng.randint(16, 128), S=S, L=_log(rng, 64, S // 8))
        if kind == "radar":
            c["gx"] = rng.choice([3, 5])
        return c
    if kind == "radar_grad":
        S = _log(rng, 4096, 32768)
        return dict(kind=kind, C=rng.randint(1, 8), P=_log(rng, 32, 512), S=S,
                    L=rng.randint(S // 16, S // 8))
    if kind == "design":
        L = rng.choice([256, 500, 777, 1024])
        return dict(kind=kind, B=_log(rng, 8, 64), L=L, n=8 * _pow2(L), C=rng.randint(1, 16),
                    P=rng.randint(32, 128), R=_log(rng, 500, 4096), T=rng.randint(4, 24))
    if kind == "ragged":
        return dict(kind=kind, jobs=_log(rng, 6, 60), shapes=rng.randint(100, 10 ** 6))
    if kind == "conv1d":
        return dict(kind=kind, rows=rng.randint(1, 16), N=_log(rng, 20000, 1048576),
                    L=_log(rng, 17, 513), mode=rng.choice(["full", "same", "valid"]))
    if kind == "fft":
        op = rng.choice(["fft", "ifft", "rfft"])
        if rng.random() < 0.4:  # along a strided axis
            n = rng.choice([64, 100, 128, 256, 512])
            return dict(kind=kind, a=rng.randint(1, 16), rows=0, n=n, cols=_log(rng, 500, 8001),
                        op="fft" if op == "rfft" else op)
        n = rng.choice([256, 1024, 4096, 8192, 16384, 65536, 1048576, _log(rng, 300, 5000),
                        _log(rng, 300, 5000)])
        top = (1 << 24) // n
        return dict(kind=kind, a=1, rows=_log(rng, max(1, top // 64), top), n=n, cols=1, op=op)
    if kind == "cfar":
        wy, wx = rng.choice([(5, 13), (7, 21)])
        return dict(kind=kind, C=rng.randint(1, 8), Ny=rng.choice([64, 100, 128, 256, 512]),
                    Nx=_log(rng, 1000, 28673), wy=wy, wx=wx, gy=3, gx=rng.choice([3, 5]),
                    want_ba=rng.random() < 0.5)
    return dict(kind="expr", C=rng.randint(1, 16), P=rng.randint(16, 128), R=_log(rng, 500, 8001))


# ------------------------------------------------------------------ inputs
def _pow2(v, strict=False):
    r = 1
    while (r <= v) if strict else (r < v):
        r *= 2
    return r


def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(seed)


def _noise(g, *shape):
    return torch.randn(shape, dtype=torch.complex64, device=DEV, generator=g)


def _uniform(g, n, lo, hi):
    return (torch.rand(n, generator=g, device=DEV, dtype=torch.float64) * (hi - lo) + lo).tolist()


def _chirp(L, bw):
    k = torch.arange(L, dtype=torch.float64, device=DEV)
    ph = 2 * math.pi * (-bw / 2 * k + 0.5 * bw / L * k * k)
    return torch.polar(torch.ones_like(ph), ph)


def _cube(g, C, P, S, L, targets, bw=0.4):
    """Receiver noise plus point echoes of a chirp, 40 to 0 dB below the noise
    in one sample (the matched filter and the Doppler sum lift them out)."""
    x = _noise(g, C, P, S)
    lfm = _chirp(L, bw)
    p = torch.arange(P, dtype=torch.float64, device=DEV)
    where = _uniform(g, targets, 0, S - L + 1)
    speed = _uniform(g, targets, 0.1, 0.9)
    snr = _uniform(g, targets, -40, 0)
    for r, f, s in zip(where, speed, snr):
        ramp = torch.polar(torch.full_like(p, 10 ** (s / 20)), 2 * math.pi * f * p)
        x[:, :, int(r):int(r) + L] += (ramp[:, None] * lfm[None, :]).to(torch.complex64)
    return x, lfm.to(torch.complex64)


def _ragged_shapes(case):
    g = torch.Generator().manual_seed(case["shapes"])
    pick = lambda lo, hi: int(torch.randint(lo, hi + 1, (1,), generator=g))  # noqa: E731
    out = []
    for _ in range(case["jobs"]):
        C, P, S = pick(1, 8), 16 << pick(0, 4), pick(1024, 16384)
        out.append((C, P, S, pick(64, min(2048, S))))
    return out


def prepare(case, seed):
    k, g, c = case["kind"], _gen(seed), case
    if k == "fft_conv":
        x, w = _cube(g, c["C"], c["P"], c["S"], c["L"], 3, 0.5)
        return dict(case=c, x=x, w=w * torch.hamming_window(c["L"], False, device=DEV))
    if k == "radar":
        x, w = _cube(g, c["C"], c["P"], c["S"], c["L"], 20)
        pipe = mx.FusedRadarPipeline(c["C"], c["P"], c["S"], c["L"], guard=(3, c["gx"]))
        pipe.set_waveform(w)
        return dict(case=c, x=x, pipe=pipe)
    if k == "stages":
        x, w = _cube(g, c["C"], c["P"], c["S"], c["L"], 10)
        return dict(case=c, x=x, w=w, pipe=mx.RadarPipeline(c["P"], c["S"], c["L"], c["C"]))
    if k == "radar_grad":
        C, P, S, L = c["C"], c["P"], c["S"], c["L"]
        x, _ = _cube(g, C, P, S, L, 20)
        phi = (torch.rand(L, generator=g, device=DEV) * 2 * math.pi).requires_grad_()
        nd, R = _pow2(P - 2), S - L + 1
        cells = [(int(f * nd), int(r * R)) for f, r in zip(_uniform(g, 20, 0, 1), _uniform(g, 20, 0, 1))]
        wmap = ag.contrast_weights(nd, R, cells, C, device=DEV)
        return dict(case=c, x=x, phi=phi, nd=nd, wmap=wmap, one=torch.ones(L, device=DEV),
                    plan=ops.PulseCompressionPlan(S, L, _pow2(S)))
    if k == "design":
        C, P, R, T = c["C"], c["P"], c["R"], c["T"]
        phi = (torch.rand((c["B"], c["L"]), generator=g, device=DEV) * 2 * math.pi).requires_grad_()
        taps = torch.hamming_window(P, False, device=DEV).requires_grad_()
        x = _noise(g, C, P, R)
        p = torch.arange(P, dtype=torch.float64, device=DEV)
        nd, tg = _pow2(P), []
        for ch, r, f, a in zip(*(_uniform(g, T, *lim) for lim in ((0, C), (0, R), (0, nd), (5, 50)))):
            x[int(ch), :, int(r)] += torch.polar(torch.full_like(p, a),
                                                 2 * math.pi * int(f) * p / nd).to(torch.complex64)
            tg.append((int(ch), int(r), int(f)))
        return dict(case=c, phi=phi, taps=taps, x=x, nd=nd,
                    targets=torch.tensor(tg, dtype=torch.int32, device=DEV))
    if k == "ragged":
        jobs = [_cube(g, C, P, S, L, 5, 0.5) for C, P, S, L in _ragged_shapes(c)]
        return dict(case=c, batch=mx.ragged.RaggedBatch(jobs))
    if k == "conv1d":
        return dict(case=c, x=_noise(g, c["rows"], c["N"]), f=_noise(g, c["L"]))
    if k == "fft":
        if c["rows"]:
            x = _noise(g, c["rows"], c["n"])
            x = x.real.contiguous() if c["op"] == "rfft" else x
        else:
            x = _noise(g, c["a"], c["n"], c["cols"])
        return dict(case=c, x=x)
    if k == "cfar":
        pw = torch.empty((c["C"], c["Ny"], c["Nx"]), device=DEV).exponential_(generator=g)
        for y, xx, s in zip(_uniform(g, 200, 0, c["Ny"]), _uniform(g, 200, 0, c["Nx"]), _uniform(g, 200, 5, 40)):
            pw[:, int(y), int(xx)] += 10 ** (s / 10)
        return dict(case=c, pw=pw)
    x = _noise(g, c["C"], c["P"], c["R"])
    nrm = torch.randint(20, 57, x.shape, generator=g, device=DEV).float()
    ba = torch.rand(x.shape, generator=g, device=DEV) * 0.4
    return dict(case=c, x=x, nrm=nrm, ba=ba, dets=torch.empty(x.shape, dtype=torch.int32, device=DEV))


# --------------------------------------------------------------- one pass
def run(state):
    s, c = state, state["case"]
    k = c["kind"]
    if k == "fft_conv":
        return mx.fft_conv(s["x"], s["w"], c["n"])
    if k == "radar":
        dets = s["pipe"].step(s["x"])
        return dict(dets=dets, y=s["pipe"].y)
    if k == "stages":
        p = s["pipe"]
        p.GetInputView()[:, :, :c["S"]].copy_(s["x"])
        p.GetwaveformView()[:c["L"]].copy_(s["w"])
        p.run()
        return dict(dets=p.GetDetections(), ba=p.GetBackgroundAverages(), pw=p.xPow)
    if k == "radar_grad":
        w = torch.polar(s["one"], s["phi"])
        pw = ag.radar_power(w, s["x"], s["plan"], s["nd"])
        loss = ag.weighted_power_sum(pw, s["wmap"])
        (gphi,) = torch.autograd.grad(loss, s["phi"])
        return dict(loss=loss.detach(), gphi=gphi)
    if k == "design":
        loss = ag.design_loss(s["phi"], s["taps"], s["x"], s["targets"], c["n"], s["nd"])
        gphi, gtaps = torch.autograd.grad(loss, (s["phi"], s["taps"]))
        return dict(loss=loss.detach(), gphi=gphi, gtaps=gtaps)
    if k == "ragged":
        return s["batch"].execute()
    if k == "conv1d":
        return mx.conv1d(s["x"], s["f"], c["mode"], method="fft")
    if k == "fft":
        axis = -1 if c["rows"] else 1
        return dict(fft=mx.fft, ifft=mx.ifft, rfft=mx.rfft)[c["op"]](s["x"], c["n"], axis)
    if k == "cfar":
        dets, ba, _ = mx.cfar(s["pw"], (c["wy"], c["wx"]), (c["gy"], c["gx"]), 1e-5,
                              want_ba=c["want_ba"])
        return dict(dets=dets, ba=ba) if c["want_ba"] else dets
    n = E.wrap(s["nrm"])
    return E.run(s["dets"], E.abs2(s["x"]) > n * (E.pow(1e-5, -1.0 / n) - 1.0) * s["ba"])


# ------------------------------------------------------------------- work
def _fft_flops(n):
    return 5 * n * math.log2(max(2, n))


def _pc_flops(rows, R, L):
    # overlap-save: a forward and an inverse transform per lag kept, of
    # blocks not much longer than twice the waveform
    return rows * R * (10 * math.log2(2 * L) + 6)


def work(case):
    k, c = case["kind"], case
    if k == "fft_conv":
        rows = c["C"] * c["P"]
        return dict(bytes=8 * (rows * (c["S"] + c["n"]) + c["L"]), flops=_pc_flops(rows, c["n"], c["L"]))
    if k in ("radar", "stages"):
        C, P, S, L = c["C"], c["P"], c["S"], c["L"]
        R, nd = S - L + 1, _pow2(P - 2) if k == "radar" else _pow2(P, True)
        cells = C * nd * R
        flops = _pc_flops(C * P, R, L) + C * R * _fft_flops(nd) + cells * 20
        # radar: samples in, compressed cube and detections out; stages: the
        # copy of the new samples, then detections, averages and power out
        out = 8 * C * P * R + 4 * cells if k == "radar" else 8 * C * P * S + 12 * cells
        return dict(bytes=8 * C * P * S + out, flops=flops)
    if k == "radar_grad":
        C, P, S, L = c["C"], c["P"], c["S"], c["L"]
        R, nd = S - L + 1, _pow2(P - 2)
        # the cube is read forward and again for the waveform's gradient
        return dict(bytes=16 * C * P * S + 4 * nd * R,
                    flops=3 * _pc_flops(C * P, R, L) / 2 + 3 * C * R * _fft_flops(nd))
    if k == "design":
        B, n = c["B"], 2 * _pow2(c["L"])
        nd, cells = _pow2(c["P"]), c["C"] * c["R"]
        return dict(bytes=8 * cells * c["P"] + 8 * B * c["L"],
                    flops=B * 6 * _fft_flops(n) + cells * (_fft_flops(nd) + 3 * nd))
    if k == "ragged":
        b = f = 0
        for C, P, S, L in _ragged_shapes(c):
            R, nd = S - L + 1, _pow2(P)
            b += 8 * C * P * S + 8 * L + 4 * C * nd * R
            f += _pc_flops(C * P, R, L) + C * R * _fft_flops(nd)
        return dict(bytes=b, flops=f)
    if k == "conv1d":
        n = c["N"] + dict(full=c["L"] - 1, same=0, valid=1 - c["L"])[c["mode"]]
        return dict(bytes=8 * c["rows"] * (c["N"] + n), flops=_pc_flops(c["rows"], n, c["L"]))
    if k == "fft":
        rows = c["rows"] or c["a"] * c["cols"]
        half = 0.5 if c["op"] == "rfft" else 1.0
        return dict(bytes=half * 16 * rows * c["n"], flops=half * rows * _fft_flops(c["n"]))
    if k == "cfar":
        cells = c["C"] * c["Ny"] * c["Nx"]
        return dict(bytes=cells * (12 if c["want_ba"] else 8), flops=cells * 20)
    cells = c["C"] * c["P"] * c["R"]
    return dict(bytes=cells * 20, flops=cells * 10)


# ------------------------------------------------- the same in 64 bits
def _hamming64(L):
    k = torch.arange(L, dtype=torch.float64, device=DEV)
    return 0.54 - 0.46 * torch.cos(2 * math.pi * k / (L - 1))


def _compress64(x, w, R, n):
    """Rows of x against the windowed unit-energy waveform, lags 0..R-1."""
    w = w.to(torch.complex128) * _hamming64(w.shape[0])
    w = w / w.abs().square().sum().sqrt()
    return torch.fft.ifft(torch.fft.fft(x.to(torch.complex128), n) * torch.fft.fft(w, n).conj())[..., :R]


def _cancel64(y, rows):
    """[1, -2, 1] along pulses of [P, R]; "valid" rows or all ("same")."""
    z = torch.nn.functional.pad(torch.view_as_real(y), (0, 0, 0, 0, 1, 1))
    z = torch.view_as_complex(z)
    t = z[:-2] - 2 * z[1:-1] + z[2:]
    return t[1:-1] if rows == "valid" else t


def _box64(pw, wy, wx, gy, gx):
    """Training-cell sums and in-bounds counts of a [Ny, Nx] map."""
    m = torch.ones((wy, wx), dtype=torch.float64, device=DEV)
    m[wy // 2 - gy // 2:wy // 2 + gy // 2 + 1, wx // 2 - gx // 2:wx // 2 + gx // 2 + 1] = 0
    H, W = pw.shape
    pad = torch.nn.functional.pad(pw, (wx // 2, wx // 2, wy // 2, wy // 2))
    one = torch.nn.functional.pad(torch.ones_like(pw), (wx // 2, wx // 2, wy // 2, wy // 2))
    s, n = torch.zeros_like(pw), torch.zeros_like(pw)
    for i, j in m.nonzero().tolist():
        s += pad[i:i + H, j:j + W]
        n += one[i:i + H, j:j + W]
    return s, n


def exact(case, seed):
    k, c = case["kind"], case
    s = prepare(case, seed) if k not in ("radar", "stages", "radar_grad", "ragged") else None
    g = _gen(seed)
    if k == "fft_conv":
        x, w = s["x"].to(torch.complex128), s["w"].to(torch.complex128)
        return torch.fft.ifft(torch.fft.fft(x, c["n"]) * torch.fft.fft(w, c["n"]).conj())
    if k == "radar":
        x, w = _cube(g, c["C"], c["P"], c["S"], c["L"], 20)
        return dict(dets=None, y=_compress64(x, w, c["S"] - c["L"] + 1, _pow2(c["S"])))
    if k == "stages":
        x, w = _cube(g, c["C"], c["P"], c["S"], c["L"], 10)
        P, R, nd = c["P"], c["S"] - c["L"] + 1, _pow2(c["P"], True)
        y = _compress64(x, w, R, _pow2(c["S"]))
        h = torch.ones(P, dtype=torch.float64, device=DEV)
        h[:P - 2] = _hamming64(P - 2)
        pw = torch.stack([torch.fft.fft(_cancel64(ch, "same") * h[:, None], nd, 0).abs().square() for ch in y])
        ba = torch.zeros((c["C"], nd + 4, R + 12), dtype=torch.float64, device=DEV)
        for ch in range(c["C"]):
            sm, n = _box64(pw[ch], 5, 13, 3, 3)
            ba[ch, 2:nd + 2, 6:R + 6] = sm / n
        return dict(dets=None, ba=ba, pw=pw)
    if k == "radar_grad":
        st = prepare(case, seed)
        P, S, L, nd = c["P"], c["S"], c["L"], st["nd"]
        phi = st["phi"].detach().double().requires_grad_()
        h, wm = _hamming64(P - 2)[:, None], st["wmap"].double()
        loss, gphi = 0.0, torch.zeros_like(phi)
        for ch in range(c["C"]):
            y = _compress64(st["x"][ch], torch.polar(torch.ones_like(phi), phi), S - L + 1, _pow2(S))
            z = torch.fft.fft(_cancel64(y, "valid") * h, nd, 0)
            part = ((z.real.square() + z.imag.square()) * wm).sum()
            gphi += torch.autograd.grad(part, phi)[0]
            loss += float(part.detach())
            del y, z, part
        return dict(loss=torch.tensor(loss, dtype=torch.float64), gphi=gphi)
    if k == "design":
        phi, taps = (s[v].detach().double().requires_grad_() for v in ("phi", "taps"))
        L, nd, n, ml, q = c["L"], s["nd"], c["n"], 2, 8
        z = torch.polar(torch.ones_like(phi), phi)
        r = torch.fft.ifft(torch.fft.fft(z, n).abs().square()).abs().square()
        isl = (r.sum(1) - r[:, 0]) / r[:, 0]
        t = s["targets"].long()
        col = s["x"][t[:, 0], :, t[:, 1]].to(torch.complex128)
        pw = torch.fft.fft(col * taps, nd).abs().square()
        d = (torch.arange(nd, device=DEV)[None, :] - t[:, 2:]) % nd
        side = (torch.minimum(d, nd - d) > ml).double()
        top = pw.detach().max()
        psl = ((pw / top).pow(q) * side).sum(1).pow(1 / q) * top / pw.gather(1, t[:, 2:])[:, 0]
        loss = isl.mean() + psl.mean()
        gphi, gtaps = torch.autograd.grad(loss, (phi, taps))
        return dict(loss=loss.detach(), gphi=gphi, gtaps=gtaps)
    if k == "ragged":
        out = []
        for C, P, S, L in _ragged_shapes(c):
            x, w = _cube(g, C, P, S, L, 5, 0.5)
            y = _compress64(x, w, S - L + 1, _pow2(S)) * _hamming64(P)[:, None]
            out.append(torch.fft.fft(y, _pow2(P), 1).abs().square())
        return out
    if k == "conv1d":
        x, f = s["x"].to(torch.complex128), s["f"].to(torch.complex128)
        N, L = c["N"], c["L"]
        n = _pow2(N + L - 1)
        full = torch.fft.ifft(torch.fft.fft(x, n) * torch.fft.fft(f, n))[:, :N + L - 1]
        lo, num = dict(full=(0, N + L - 1), same=((L - 1) // 2, N), valid=(L - 1, N - L + 1))[c["mode"]]
        return full[:, lo:lo + num].contiguous()
    if k == "fft":
        x = s["x"].to(torch.float64 if c["op"] == "rfft" else torch.complex128)
        f = dict(fft=torch.fft.fft, ifft=torch.fft.ifft, rfft=torch.fft.rfft)[c["op"]]
        return f(x, c["n"], -1 if c["rows"] else 1)
    if k == "cfar" and c["want_ba"]:
        ba = [torch.div(*_box64(m.double(), c["wy"], c["wx"], c["gy"], c["gx"])) for m in s["pw"]]
        return dict(dets=None, ba=torch.stack(ba))
    return None
