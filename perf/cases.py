"""The work a user of the PESQ loss has it do, as cases that can be timed and checked.

A case is a dict of plain values.  ``kind`` says which public entry point it
goes through:

``loss``
    ``PesqLossTriton``: an evaluation (``call`` = ``mos``, no gradient), a
    training step (``call`` = ``loss``: the loss and the gradient of its sum
    with respect to the degraded signal, or to both) or the whole step as one
    graph replay (``call`` = ``graph``: new inputs copied in, replayed).
``lfilter``
    ``HipIIR``: a band pass of even order and its adjoint.
``resample``
    ``HipResample`` and its adjoint.
``spectral``
    ``HipStftBark``: the Bark spectrogram and its adjoint.
``chain``
    ``HipPesqChain``: the distances of two Bark spectrograms and their adjoint.
"""

import functools
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "triton-pesq_amd"))

from torch_pesq import PesqLossTriton  # noqa: E402
from torch_pesq.hip_ops.chain import HipPesqChain  # noqa: E402
from torch_pesq.hip_ops.iir import HipIIR  # noqa: E402
from torch_pesq.hip_ops.resample import HipResample  # noqa: E402
from torch_pesq.hip_ops.spectral import HipStftBark  # noqa: E402

FACTOR = 0.5
PESQ_STFT = (512, 512, 256)  # n_fft, win_length, hop_length


def _loss(name, call, rate, batch, samples, grad, noise, stft=PESQ_STFT):
    case = {"kind": "loss", "call": call, "rate": rate, "batch": batch, "samples": samples, "grad": grad,
            "noise": noise, "n_fft": stft[0], "win_length": stft[1], "hop": stft[2]}
    return dict(case, name=name) if name else case


def listed():
    return [
        # one second of speech scored in a loop, file by file: the smallest call
        _loss("mos_1x1s_16k", "mos", 16000, 1, 16000, "none", "white"),
        # the usual training step of a speech enhancer at 16 kHz, through autograd
        _loss("loss_8x8s_16k", "loss", 16000, 8, 128000, "deg", "white"),
        # the same step as one graph, new inputs each time
        _loss("graph_8x8s_16k", "graph", 16000, 8, 128000, "deg", "white"),
        # training on music-rate material: the 441:160 resampler before the pipeline
        _loss("loss_16x4s_44k", "loss", 44100, 16, 176400, "deg", "pink"),
        # few, long recordings: rows of many scan blocks
        _loss("loss_4x60s_16k", "loss", 16000, 4, 960000, "deg", "clip"),
        # a full batch of a large training run at 48 kHz: the largest call
        _loss("loss_256x4s_48k", "loss", 48000, 256, 192000, "deg", "mixed"),
        # scoring a folder of utterances cut to one odd length, 22.05 kHz, no gradient
        _loss("mos_37x7s_22k", "mos", 22050, 37, 161185, "none", "white"),
        # telephone speech (8 kHz, upsampled), both inputs from networks
        _loss("loss_both_24x5s_8k", "loss", 8000, 24, 42377, "both", "pink"),
        # another STFT geometry (25 ms windows, 10 ms hop): the stage by stage path
        _loss("loss_16x4s_400_160", "loss", 16000, 16, 64000, "deg", "white", (512, 400, 160)),
        # the stand-alone recursive filter inside a network, order 16, ragged rows
        {"name": "lfilter_16_24x10s", "kind": "lfilter", "order": 16, "lo": 325, "hi": 3250, "batch": 24, "samples": 160001},
        # augmentation: up to 44.1 kHz and the adjoint back
        {"name": "resample_16k_44k_32x4s", "kind": "resample", "orig": 16000, "new": 44100, "batch": 32, "samples": 65537},
        # Bark features of another model: longer windows, quarter hop
        {"name": "spectral_1024_32x4s", "kind": "spectral", "n_fft": 1024, "win_length": 1024, "hop": 256, "batch": 32, "samples": 64123},
    ]


def _spread(rng, low, high):
    return math.exp(rng.uniform(math.log(low), math.log(high)))


def draw(rng):
    kind = rng.choice(["loss"] * 6 + ["general", "lfilter", "resample", "spectral", "chain"])
    noise = rng.choice(["white", "pink", "clip", "mixed"])
    if kind == "loss":
        call = rng.choice(["loss", "loss", "loss", "mos", "graph"])
        rate = rng.choice([16000, 16000, 16000, 8000, 22050, 32000, 44100, 48000])
        seconds = _spread(rng, 1.0, 60.0)
        batch = max(1, min(256, int(_spread(rng, 1.0, min(256.0, 1000.0 / seconds)))))
        samples = int(seconds * rate) + rng.randrange(256)
        grad = "none" if call == "mos" else rng.choice(["deg", "deg", "both"])
        if grad == "both":
            batch = max(1, batch // 2)
        return _loss(None, call, rate, batch, samples, grad, noise)
    batch, seconds = int(_spread(rng, 1.0, 65.0)), _spread(rng, 1.0, 8.0)
    if kind == "general":
        stft = rng.choice([(256, 256, 128), (512, 400, 160), (512, 400, 256), (512, 512, 200), (1024, 1024, 512)])
        samples = int(seconds * 16000) + rng.randrange(256)
        # rows whose last frame ends before the tail's 15 sample ramp
        while (samples + samples % 256 - stft[0]) // stft[2] * stft[2] + stft[0] > samples - 15:
            samples += 1
        return _loss(None, "loss", 16000, batch, samples, "deg", noise, stft)
    if kind == "lfilter":
        return {"kind": "lfilter", "order": rng.choice([2, 4, 10, 16]), "lo": 325, "hi": 3250, "batch": batch, "samples": int(seconds * 16000) + rng.randrange(16)}
    if kind == "resample":
        orig, new = rng.choice([(16000, 44100), (16000, 48000), (48000, 44100), (44100, 16000), (48000, 16000), (8000, 16000), (22050, 16000)])
        return {"kind": "resample", "orig": orig, "new": new, "batch": batch, "samples": int(seconds * orig) + rng.randrange(256)}
    if kind == "spectral":
        n_fft, win, hop = rng.choice([(256, 256, 64), (256, 256, 128), (512, 400, 160), (512, 512, 256), (1024, 800, 320), (1024, 1024, 256)])
        return {"kind": "spectral", "n_fft": n_fft, "win_length": win, "hop": hop, "batch": batch, "samples": int(seconds * 16000) + rng.randrange(256)}
    return {"kind": "chain", "batch": batch, "frames": int(_spread(rng, 60.0, 4000.0))}


# -- inputs -------------------------------------------------------------------


def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _uniform(g, batch, low, high):
    return low + (high - low) * torch.rand(batch, 1, generator=g, device="cuda")


def _speech(g, batch, samples, rate, harmonic_only):
    """Voiced speech: harmonics of a vibrato f0 under three formants, syllables
    of 250 ms of which a fifth are silent, a recording's noise floor, RMS 0.05.
    Rows of ``harmonic_only`` have neither formants nor syllables."""

    t = torch.arange(samples, device="cuda", dtype=torch.float64)[None] / rate
    f0 = _uniform(g, batch, 100.0, 250.0).double()
    vib = _uniform(g, batch, 0.0, 1.0).double()
    # cycles of f0 (1 + 0.1 sin(2 pi (5 t + vib)))
    cycles = f0 * (t - 0.1 * torch.cos(2 * math.pi * (5.0 * t + vib)) / (10 * math.pi))
    cycles = (cycles - cycles.floor()).float()
    signal = torch.zeros(batch, samples, device="cuda")
    for k in range(1, 25):
        freq = k * f0.float()
        amp = sum(1.0 / (1.0 + ((freq - fc) / bw) ** 2) for fc, bw in ((500, 80), (1500, 120), (2500, 160)))
        amp = torch.where(harmonic_only, torch.ones_like(amp), amp + 0.02) / k
        amp = amp * (freq * 1.1 < 0.45 * rate)
        signal += amp * torch.sin((2 * math.pi) * torch.frac(k * cycles))
    syllable = (t[0] * 4.0).long()
    on = (torch.rand(batch, int(syllable[-1]) + 1, generator=g, device="cuda") >= 0.2).float()
    envelope = (0.5 - 0.5 * torch.cos(8 * math.pi * t)).float() * on[:, syllable]
    signal = signal * torch.where(harmonic_only, torch.ones_like(envelope), envelope)
    signal = signal * (0.05 / signal.square().mean(1, keepdim=True).sqrt().clamp(min=1e-6))
    return signal + 3e-5 * torch.randn(batch, samples, generator=g, device="cuda")


def _noise(g, batch, samples, pink):
    noise = torch.randn(batch, samples, generator=g, device="cuda")
    if pink:
        spec = torch.fft.rfft(noise)
        freq = torch.arange(spec.shape[1], device="cuda").clamp(min=1).float()
        noise = torch.fft.irfft(spec / freq.sqrt(), samples)
        noise = noise / noise.square().mean(1, keepdim=True).sqrt()
    return noise


def _signals(case, seed):
    """Reference and degraded speech of a ``loss`` case."""

    g = _generator(seed)
    batch, samples, mixed = case["batch"], case["samples"], case["noise"] == "mixed"
    harmonic = _uniform(g, batch, 0.0, 1.0) < (0.25 if mixed else 0.0)
    ref = _speech(g, batch, samples, case["rate"], harmonic)
    if case["noise"] == "white":
        snr = _uniform(g, batch, 0.0, 20.0)
    elif mixed:
        snr = _uniform(g, batch, -5.0, 20.0)
    else:
        snr = torch.full((batch, 1), 5.0 if case["noise"] == "pink" else 0.0, device="cuda")
    noise = _noise(g, batch, samples, case["noise"] in ("pink", "clip"))
    deg = ref + noise * (0.05 * 10 ** (-snr / 20.0))
    if case["noise"] == "clip":
        peak = 0.8 * deg.abs().amax(1, keepdim=True)
        deg = torch.minimum(torch.maximum(deg, -peak), peak)
    if mixed:
        gain = 10 ** (_uniform(g, batch, -20.0, 6.0) / 20.0)
        deg = deg * torch.where(_uniform(g, batch, 0.0, 1.0) < 0.1, gain, torch.ones_like(gain))
    return ref.contiguous(), deg.contiguous()


# -- modules, as a program keeps them -----------------------------------------


@functools.lru_cache(maxsize=8)
def _pesq(rate, n_fft, win_length, hop):
    return PesqLossTriton(FACTOR, sample_rate=rate, n_fft=n_fft, win_length=win_length, hop_length=hop).cuda()


def _model(case):
    return _pesq(case["rate"], case["n_fft"], case["win_length"], case["hop"])


def _band_pass(order, lo, hi, rate=16000):
    """Butterworth band pass of even ``order``: (b, a) by the bilinear transform."""

    half = order // 2
    w1, w2 = (2 * rate * math.tan(math.pi * f / rate) for f in (lo, hi))
    width, centre = w2 - w1, math.sqrt(w1 * w2)
    proto = np.exp(1j * math.pi * (2 * np.arange(half) + half + 1) / (2 * half))
    shifted = proto * width / 2
    root = np.sqrt(shifted**2 - centre**2 + 0j)
    analog = np.concatenate([shifted + root, shifted - root])
    poles = (2 * rate + analog) / (2 * rate - analog)
    a = np.real(np.poly(poles))
    b = np.real(np.poly(np.concatenate([np.ones(half), -np.ones(half)])))
    z = np.exp(2j * math.atan(centre / (2 * rate)))  # unit gain at the centre
    gain = abs(np.polyval(a, z) / np.polyval(b, z))
    return b * gain, a


@functools.lru_cache(maxsize=8)
def _lfilter(order, lo, hi):
    return HipIIR(*_band_pass(order, lo, hi)).cuda()


@functools.lru_cache(maxsize=8)
def _resampler(orig, new):
    return HipResample(orig, new).cuda()


@functools.lru_cache(maxsize=8)
def _spectral(n_fft, win_length, hop):
    bank = _pesq(16000, n_fft, n_fft, n_fft // 2).fbank
    return HipStftBark(torch.hann_window(win_length), bank.fbank, bank.pow_dens_correction, n_fft, hop).cuda()


@functools.lru_cache(maxsize=1)
def _chain():
    model = _pesq(16000, *PESQ_STFT)
    return HipPesqChain(model.loudness.threshs, model.loudness.exp, model.fbank.width_bark, float(model.fbank.total_width)).cuda()


def prepare(case, seed):
    kind = case["kind"]
    if kind == "loss":
        ref, deg = _signals(case, seed)
        ref.requires_grad_(case["grad"] == "both")
        deg.requires_grad_(case["grad"] != "none")
        state = {"case": case, "model": _model(case), "ref": ref, "deg": deg}
        if case["call"] == "graph":
            state["step"] = state["model"].graphed_step(ref, deg)
            state["ref"], state["deg"] = ref.detach(), deg.detach()
        return state
    g = _generator(seed)
    if kind == "chain":
        # Bark spectra of speech at the aligned level: powers over many decades
        # around the thresholds, the degraded ones correlated with the reference
        model = _chain()
        shape = (case["batch"], case["frames"], model.threshs.shape[0])
        level = 9.0 * torch.rand(case["batch"], case["frames"], 1, generator=g, device="cuda")
        ref = model.threshs * 10 ** (level - 2.0 + torch.randn(shape, generator=g, device="cuda"))
        deg = ref * 10 ** (0.4 * torch.randn(shape, generator=g, device="cuda")) + 10.0 * model.threshs
        weights = 0.1 + torch.rand(2, case["batch"], generator=g, device="cuda")
        return {"case": case, "model": model, "ref": ref, "x": deg.requires_grad_(), "g": weights}
    if kind == "lfilter":
        module, rate = _lfilter(case["order"], case["lo"], case["hi"]), 16000
    elif kind == "resample":
        module, rate = _resampler(case["orig"], case["new"]), case["orig"]
    else:
        module, rate = _spectral(case["n_fft"], case["win_length"], case["hop"]), 16000
    x = _speech(g, case["batch"], case["samples"], rate, torch.zeros(case["batch"], 1, dtype=torch.bool, device="cuda"))
    x = (x + 0.005 * torch.randn(x.shape, generator=g, device="cuda")).contiguous()
    if kind == "lfilter":
        shape = x.shape
    elif kind == "resample":
        shape = (case["batch"], _resampled(case["samples"], case["orig"], case["new"]))
    else:
        shape = (case["batch"], 1 + (case["samples"] - case["n_fft"]) // case["hop"], 49)
    upstream = torch.randn(shape, generator=g, device="cuda")
    return {"case": case, "model": module, "x": x.requires_grad_(), "g": upstream}


def run(state):
    case, model = state["case"], state["model"]
    kind = case["kind"]
    if kind == "loss":
        ref, deg = state["ref"], state["deg"]
        if case["call"] == "mos":
            return {"mos": model.mos(ref, deg)}
        if case["call"] == "graph":
            step = state["step"]
            static_ref, static_deg = step.inputs()
            with torch.no_grad():
                static_ref.copy_(ref)
                static_deg.copy_(deg)
            step.replay()
            loss, g_ref, g_deg = step.outputs()
            out = {"loss": loss, "g_deg": g_deg}
            return dict(out, g_ref=g_ref) if case["grad"] == "both" else out
        loss = model(ref, deg)
        if case["grad"] == "both":
            g_ref, g_deg = torch.autograd.grad(loss.sum(), (ref, deg))
            return {"loss": loss, "g_deg": g_deg, "g_ref": g_ref}
        (g_deg,) = torch.autograd.grad(loss.sum(), deg)
        return {"loss": loss, "g_deg": g_deg}
    if kind == "chain":
        symm, asymm = model(state["ref"], state["x"])
        (g_x,) = torch.autograd.grad((symm, asymm), state["x"], (state["g"][0], state["g"][1]))
        return {"symm": symm, "asymm": asymm, "g_x": g_x}
    y = model(state["x"])
    (g_x,) = torch.autograd.grad(y, state["x"], state["g"])
    return {"y": y, "g_x": g_x}


# -- what a pass cannot do without --------------------------------------------


def _resampled(samples, orig, new):
    step = math.gcd(orig, new)
    return int(np.ceil(np.float32(new // step * samples / (orig // step))))


def work(case):
    kind, batch = case["kind"], case["batch"]
    if kind == "chain":
        values = batch * case["frames"] * 49
        return {"bytes": 4 * 3 * values, "flops": 300 * values}
    samples = case["samples"]
    if kind == "lfilter":
        # b and a of each order, forward and adjoint
        return {"bytes": 4 * 4 * batch * samples, "flops": 2 * 2 * (2 * case["order"] + 1) * batch * samples}
    if kind == "resample":
        out = batch * _resampled(samples, case["orig"], case["new"])
        taps = 2 * 6 / 0.99 * max(1.0, case["orig"] / case["new"])
        return {"bytes": 4 * 2 * (batch * samples + out), "flops": 2 * 2 * taps * out}
    n_fft = case["n_fft"]
    transform = 2.5 * n_fft * math.log2(n_fft) + 4 * n_fft
    if kind == "spectral":
        frames = batch * (1 + (samples - n_fft) // case["hop"])
        return {"bytes": 4 * (2 * batch * samples + 2 * 49 * frames), "flops": 3 * transform * frames}
    grads = {"none": 0, "deg": 1, "both": 2}[case["grad"]]
    low = _resampled(samples, case["rate"], 16000)
    frames = 1 + (low + low % 256 - n_fft) // case["hop"]
    taps = 0.0 if case["rate"] == 16000 else 2 * 6 / 0.99 * max(1.0, case["rate"] / 16000)
    filters = low * 2 * (2 * 10 + 1 + 2 * 2 + 1)
    signal = 2 * taps * low + filters + frames * (transform + 100 * 49)
    adjoint = 2 * taps * low + filters + frames * (2 * transform + 100 * 49)
    return {"bytes": 4 * batch * ((2 + grads) * samples + 1), "flops": batch * (2 * signal + grads * adjoint)}


def tolerance(case):
    """About four times the largest errors against ``exact`` seen over the ranges."""

    kind = case["kind"]
    if kind == "loss":
        if case["grad"] == "none":
            return {"rel": 1.2e-6, "max": 4e-6}
        # the float32 transforms of the fused path, and terms near the chain's
        # clamps and thresholds (more of them in the reference's gradient)
        return {"rel": 6e-5, "max": 4e-3} if case["grad"] == "deg" else {"rel": 9e-4, "max": 2e-2}
    if kind == "lfilter" and case["order"] > 12:
        # the realisation in sections against the difference equation itself
        return {"rel": 1.1e-5, "max": 6.5e-5}
    if kind == "chain":
        return {"rel": 2e-7, "max": 1e-6}
    if kind == "spectral":
        return {"rel": 2e-7, "max": 2.2e-6}
    return {"rel": 1e-7, "max": 2.5e-7}


# -- the same in 64 bits --------------------------------------------------------


def _impulse(b, a, taps):
    """Impulse response of the difference equation b / a."""

    b, a = (np.asarray(v, dtype=np.float64) for v in (b, a))
    h = np.zeros(taps + len(a) - 1)
    back = -(a[1:] / a[0])[::-1]
    order = len(a) - 1
    for n in range(taps):
        h[n + order] = np.dot(back, h[n : n + order]) + (b[n] / a[0] if n < len(b) else 0.0)
    return torch.from_numpy(h[order:].copy()).cuda()


def _convolved(x, h):
    size = 1 << (x.shape[1] + h.shape[0] - 1).bit_length()
    return torch.fft.irfft(torch.fft.rfft(x, size) * torch.fft.rfft(h, size), size)[:, : x.shape[1]]


def _resampled64(x, module, out_samples):
    """The polyphase form of the filter bank: one dot product per output."""

    orig, width, bank = module.orig_step, module.width, module.kernel.double()
    padded = torch.nn.functional.pad(x, (width, width + orig))
    y = padded.unfold(1, bank.shape[1], orig).contiguous() @ bank.t()
    return y.reshape(x.shape[0], -1)[:, :out_samples]


def _bark64(x, window, fbank, corr, n_fft, hop):
    left = (n_fft - window.shape[0]) // 2
    full = torch.nn.functional.pad(window, (left, n_fft - window.shape[0] - left))
    spec = torch.fft.rfft(x.unfold(1, n_fft, hop) * full)
    power = spec.real.square() + spec.imag.square()
    return (power[..., 1:-1] @ fbank[:, 1:].t()) * corr


def _chain64(ref, deg, th, ex, width, total, sl=0.1866055):
    def audible(spec, factor):
        return (spec * (spec > factor * th)).sum(-1)

    def loudness(spec):
        loud = (2 * th) ** ex * ((0.5 + 0.5 * torch.maximum(spec, th) / th) ** ex - 1.0)
        return sl * torch.where(spec <= th, torch.zeros_like(loud), loud)

    heard = (audible(ref, 100.0) >= 1e7)[..., None]
    means = [(s * ((s > 100.0 * th) & heard)).mean(1) for s in (ref, deg)]
    equ_ref = ref * ((means[1] + 1000.0) / (means[0] + 1000.0)).clamp(0.01, 100.0)[:, None]
    total_ref = audible(equ_ref, 1.0)
    ratio = (total_ref + 5e3) / (audible(deg, 1.0) + 5e3)
    ratio = torch.cat([ratio[:, :1], 0.8 * ratio[:, 1:] + 0.2 * ratio[:, :-1]], 1).clamp(3e-4, 5.0)
    equ_deg = deg * ratio[..., None]
    loud_ref, loud_deg = loudness(equ_ref), loudness(equ_deg)
    diff = loud_deg - loud_ref
    dist = diff.sign() * (diff.abs() - 0.25 * torch.minimum(loud_ref, loud_deg)).clamp(min=0)
    skew = ((equ_deg + 50.0) / (equ_ref + 50.0)) ** 1.2
    skew = torch.where(skew < 3.0, torch.zeros_like(skew), skew).clamp(max=12.0)
    h = ((total_ref + 1e5) / 1e7) ** 0.04
    out = []
    for terms, p in ((width * dist, 2), (width * dist * skew, 1)):
        frame = total ** (1 - 1 / p) * terms[..., 1:].norm(p, dim=-1)
        frame = (frame.clamp(min=1e-20) / h).clamp(max=45.0)
        windows = (frame.unfold(1, 20, 10) ** 6).mean(-1) ** (1 / 6)
        out.append(windows.square().mean(1).sqrt())
    return out


def _pesq64(case, model, ref, deg):
    """Distances of a few rows, every stage in 64 bits."""

    bank, loud = model.fbank, model.loudness
    power, pre = (_impulse(*f.detach().cpu().numpy(), 8192) for f in (model.power_filter, model.pre_filter))
    ramp = torch.arange(1, 16, device="cuda", dtype=torch.float64) / 16
    barks = []
    for x in (ref, deg):
        if case["rate"] != 16000:
            x = _resampled64(x, model.resampler, _resampled(x.shape[1], case["rate"], 16000))
        samples = x.shape[1]
        energy = _convolved(x, power).square().sum(1, keepdim=True)
        x = x * (1e7 * 1.04684 * (samples + 5120) / energy).sqrt()
        ones = torch.ones(samples - 15, device="cuda", dtype=torch.float64)
        x = _convolved(x * torch.cat([ramp, ones]) * torch.cat([ones, ramp.flip(0)]), pre)
        x = torch.nn.functional.pad(x, (0, samples % 256))
        window = torch.hann_window(case["win_length"]).cuda().double()
        barks.append(_bark64(x, window, bank.fbank.double(), bank.pow_dens_correction.double().reshape(-1), case["n_fft"], case["hop"]))
    return _chain64(*barks, loud.threshs.double().reshape(-1), loud.exp.double().reshape(-1), bank.width_bark.double().reshape(-1), float(bank.total_width))


def exact(case, seed):
    kind = case["kind"]
    if kind == "loss":
        if case["batch"] * case["samples"] > 60e6:
            return None
        model = _model(case)
        rows = [t.double() for t in _signals(case, seed)]
        few = max(1, 2_000_000 // case["samples"])
        losses, moses, grads = [], [], {"ref": [], "deg": []}
        for at in range(0, case["batch"], few):
            ref, deg = (t[at : at + few].clone().requires_grad_(case["grad"] != "none") for t in rows)
            symm, asymm = _pesq64(case, model, ref, deg)
            raw = 0.1 * symm + 0.0309 * asymm
            losses.append((FACTOR * raw).detach())
            moses.append((0.999 + 4 / (1 + torch.exp(-1.3669 * (4.5 - raw) + 3.8224))).detach())
            if case["grad"] != "none":
                g_ref, g_deg = torch.autograd.grad((FACTOR * raw).sum(), (ref, deg))
                grads["ref"].append(g_ref)
                grads["deg"].append(g_deg)
        if case["call"] == "mos":
            return {"mos": torch.cat(moses)}
        out = {"loss": torch.cat(losses), "g_deg": torch.cat(grads["deg"])}
        return dict(out, g_ref=torch.cat(grads["ref"])) if case["grad"] == "both" else out
    state = prepare(case, seed)
    module, g = state["model"], state["g"].double()
    x = state["x"].detach().double().requires_grad_()
    if kind == "chain":
        loss = _pesq(16000, *PESQ_STFT)
        th, ex, width = (t.cuda().double().reshape(-1) for t in (loss.loudness.threshs, loss.loudness.exp, loss.fbank.width_bark))
        symm, asymm = _chain64(state["ref"].double(), x, th, ex, width, float(loss.fbank.total_width))
        (g_x,) = torch.autograd.grad((symm, asymm), x, (g[0], g[1]))
        return {"symm": symm.detach(), "asymm": asymm.detach(), "g_x": g_x}
    if kind == "lfilter":
        y = _convolved(x, _impulse(*_band_pass(case["order"], case["lo"], case["hi"]), 16384))
    elif kind == "resample":
        y = _resampled64(x, module, g.shape[1])
    else:
        bank = _pesq(16000, case["n_fft"], case["n_fft"], case["n_fft"] // 2).fbank
        window = torch.hann_window(case["win_length"]).cuda().double()
        y = _bark64(x, window, bank.fbank.double(), bank.pow_dens_correction.double().reshape(-1), case["n_fft"], case["hop"])
    (g_x,) = torch.autograd.grad(y, x, g)
    return {"y": y.detach(), "g_x": g_x}
