"""GPU parity of the STFT / Bark operator beyond the PESQ geometry.

``HipStftBark`` with other FFT lengths, band counts, hops and short windows
runs the general kernels of ``csrc/stft_generic.hip``; the cases follow the
reference's ``tests/test_triton_spectral.py:294-312,340-420,638-700``.

Oracle: ``oracle.pesq_oracle.stft_bark_op`` (float64 ``torch.stft``, DC
dropped, band sums), pinned against a direct float64 DFT in
``test_oracle.py``; gradients by float64 autograd through it.

Tolerance, the reference's error model for a spectrogram
(``test_triton_spectral.py:1-45``): ``|got - want| <= RTOL |want| + ATOL *
local_scale`` with the local scale the peak of the frame (forward) or of the
gradient over the frames a sample belongs to (backward); ``RTOL = 1e-5``,
``ATOL = 5e-6`` forward and ``1e-5`` backward.  The float64 FFT leaves the
float32 rounding of the outputs (about 1e-7).
"""

import numpy as np
import pytest
import torch
import torch.nn.functional as F

from oracle import pesq_oracle as O
from torch_pesq.bark import BarkScale
from torch_pesq.hip_ops.spectral import HipStftBark

pytestmark = pytest.mark.gpu

RTOL = 1e-5
ATOL_FWD = 5e-6
ATOL_BWD = 1e-5


def _module(n_fft=512, nbarks=49, hop=256, window=None):
    scale = BarkScale(n_fft // 2, nbarks)
    window = torch.hann_window(n_fft) if window is None else window
    mod = HipStftBark(window, scale.fbank, scale.pow_dens_correction, n_fft, hop).cuda()
    return mod, window, scale


def _oracle(signal, mod, window, scale, n_padded=None):
    return O.stft_bark_op(signal.double().cpu(), window, scale.fbank, scale.pow_dens_correction,
                          mod.n_fft, mod.hop_length, n_padded)


def _violation(got, want, atol, scale):
    delta = (got.double().cpu() - want).abs()
    return float((delta - (RTOL * want.abs() + atol * scale)).max())


def _frame_scale(want):
    return want.abs().amax(dim=2, keepdim=True)


def _sample_scale(grad, hop, novertaps):
    n = grad.shape[1]
    blocks = F.pad(grad.abs(), (0, (-n) % hop)).reshape(grad.shape[0], -1, hop).amax(dim=2)
    dilated = F.max_pool1d(blocks.unsqueeze(1), 2 * novertaps + 1, 1, novertaps).squeeze(1)
    return dilated.repeat_interleave(hop, dim=1)[:, :n]


def _both(mod, window, scale, signal, n_padded=None, seed=0):
    x = signal.clone().requires_grad_(True)
    got = mod(x, n_padded)
    gen = torch.Generator().manual_seed(seed)
    up = torch.randn(got.shape, generator=gen, dtype=torch.float64)
    (g_got,) = torch.autograd.grad(got, x, up.float().cuda())
    xd = signal.double().cpu().requires_grad_(True)
    want = O.stft_bark_op(xd, window, scale.fbank, scale.pow_dens_correction, mod.n_fft,
                          mod.hop_length, n_padded)
    (g_want,) = torch.autograd.grad(want, xd, up)
    return got, want.detach(), g_got, g_want


@pytest.mark.parametrize("n_fft,nbarks", [(512, 32), (256, 49), (256, 32), (1024, 49), (64, 17)])
@pytest.mark.parametrize("batch,nsamples", [(1, 4096), (3, 5003), (5, 1024)])
def test_forward_parity(n_fft, nbarks, batch, nsamples):
    mod, window, scale = _module(n_fft, nbarks)
    assert mod.general
    torch.manual_seed(nsamples + n_fft + nbarks)
    signal = torch.randn(batch, nsamples, device="cuda") * 3000.0
    got = mod(signal)
    want = _oracle(signal, mod, window, scale)
    assert got.shape == want.shape
    assert _violation(got, want, ATOL_FWD, _frame_scale(want)) <= 0.0


@pytest.mark.parametrize("n_fft,nbarks", [(512, 32), (256, 49)])
def test_backward_parity(n_fft, nbarks):
    mod, window, scale = _module(n_fft, nbarks)
    torch.manual_seed(n_fft + nbarks)
    signal = torch.randn(3, 5003, device="cuda") * 1000.0
    got, want, g_got, g_want = _both(mod, window, scale, signal, seed=3)
    assert _violation(got, want, ATOL_FWD, _frame_scale(want)) <= 0.0
    scale_s = _sample_scale(g_want, mod.hop_length, mod.novertaps)
    assert _violation(g_got, g_want, ATOL_BWD, scale_s) <= 0.0


@pytest.mark.parametrize("hop_length", [128, 600, 100, 37])
def test_hop_length_sweep(hop_length):
    mod, window, scale = _module(512, 49, hop_length)
    assert mod.general
    assert mod.novertaps == -(-512 // hop_length)
    torch.manual_seed(hop_length)
    signal = torch.randn(2, 4096, device="cuda") * 1000.0
    got, want, g_got, g_want = _both(mod, window, scale, signal, seed=hop_length)
    assert got.shape[1] == 1 + (4096 - 512) // hop_length
    assert _violation(got, want, ATOL_FWD, _frame_scale(want)) <= 0.0
    scale_s = _sample_scale(g_want, hop_length, mod.novertaps)
    assert _violation(g_got, g_want, ATOL_BWD, scale_s) <= 0.0


def test_gradient_is_zero_in_the_gaps_between_frames():
    mod, window, scale = _module(512, 49, 600)
    signal = (torch.randn(1, 3000, device="cuda") * 1000.0).requires_grad_(True)
    out = mod(signal)
    (g,) = torch.autograd.grad(out.sum(), signal)
    covered = torch.zeros(3000, dtype=torch.bool)
    for t in range(out.shape[1]):
        covered[600 * t : 600 * t + 512] = True
    assert torch.count_nonzero(g[0, ~covered.cuda()]) == 0
    assert torch.count_nonzero(g[0, covered.cuda()]) > 0


@pytest.mark.parametrize("win_length", [400, 401, 33])
def test_short_window_is_centred(win_length):
    window = torch.hann_window(win_length)
    mod, _, scale = _module(512, 49, 256, window)
    torch.manual_seed(23)
    signal = torch.randn(2, 4096, device="cuda") * 1000.0
    got, want, g_got, g_want = _both(mod, window, scale, signal, seed=win_length)
    assert _violation(got, want, ATOL_FWD, _frame_scale(want)) <= 0.0
    scale_s = _sample_scale(g_want, 256, mod.novertaps)
    assert _violation(g_got, g_want, ATOL_BWD, scale_s) <= 0.0


def test_padding_and_tail_samples():
    """Frames past the signal read zeros; samples after the last frame get no gradient."""

    mod, window, scale = _module(256, 32, 128)
    torch.manual_seed(5)
    signal = torch.randn(2, 3001, device="cuda") * 100.0
    got, want, g_got, g_want = _both(mod, window, scale, signal, n_padded=3200, seed=5)
    assert got.shape[1] == 1 + (3200 - 256) // 128
    assert _violation(got, want, ATOL_FWD, _frame_scale(want)) <= 0.0
    scale_s = _sample_scale(g_want, 128, mod.novertaps)
    assert _violation(g_got, g_want, ATOL_BWD, scale_s) <= 0.0


def test_general_path_is_deterministic_and_rows_independent():
    mod, _, _ = _module(256, 49, 100)
    signal = torch.randn(4, 6000, device="cuda").requires_grad_(True)
    a, b = mod(signal), mod(signal)
    assert torch.equal(a, b)
    assert torch.equal(mod(signal[2:3]), a[2:3])
    (g1,) = torch.autograd.grad(a.sum(), signal)
    (g2,) = torch.autograd.grad(mod(signal).sum(), signal)
    assert torch.equal(g1, g2)


def test_default_geometry_agrees_with_the_general_kernels():
    """The PESQ geometry through both kernel families (radix-4 vs radix-2)."""

    mod, window, scale = _module(512, 49, 256)
    assert not mod.general
    torch.manual_seed(9)
    signal = torch.randn(2, 8000, device="cuda") * 1000.0
    want = _oracle(signal, mod, window, scale)
    got = mod(signal)
    assert _violation(got, want, ATOL_FWD, _frame_scale(want)) <= 0.0
    mod.general = True  # route the same constants through the general kernels
    mod.table = _general_table_for(mod, window, scale)
    got2 = mod(signal)
    assert _violation(got2, want, ATOL_FWD, _frame_scale(want)) <= 0.0


def _general_table_for(mod, window, scale):
    from torch_pesq.hip_ops.spectral import _general_table

    return _general_table(mod.window, mod.starts, mod.ends, scale.pow_dens_correction,
                          mod.n_fft, mod.hop_length).cuda()


# ---------------------------------------------------------------------------
# the whole loss at other STFT geometries (PesqLossTriton(n_fft=..., ...))
# ---------------------------------------------------------------------------

GEOMETRIES = [(256, 256, 128), (512, 400, 256), (512, 512, 200), (1024, 1024, 512)]


def _oracle_constants(n_fft, win_length, hop):
    c = dict(O.constants())
    c.update(n_fft=n_fft, hop=hop, window=torch.hann_window(win_length).double(),
             fbank=O.bark_fbank(n_fft // 2, 49))
    return c


@pytest.mark.parametrize("n_fft,win_length,hop", GEOMETRIES)
def test_loss_at_other_geometries_matches_float64(n_fft, win_length, hop):
    from bench import speech_like_pair
    from torch_pesq import PesqLossTriton

    model = PesqLossTriton(0.5, sample_rate=16000, n_fft=n_fft, win_length=win_length,
                           hop_length=hop).cuda()
    assert model.general
    ref, deg = speech_like_pair(2, 24000, seed=n_fft + hop, noise=0.1)
    r = torch.from_numpy(ref).cuda().requires_grad_(True)
    d = torch.from_numpy(deg).cuda().requires_grad_(True)
    ds, da, mos, loss = model._run(r, d)
    weights = torch.tensor([0.7, -1.3], dtype=torch.float64)
    g_ref, g_deg = torch.autograd.grad(loss, [r, d], grad_outputs=weights.float().cuda())

    c = _oracle_constants(n_fft, win_length, hop)
    rd = torch.from_numpy(ref).double().requires_grad_(True)
    dd = torch.from_numpy(deg).double().requires_grad_(True)
    wds, wda = O.pipeline(rd, dd, c=c)
    wmos, wloss = O.epilogue(wds, wda, 0.5)
    (wloss * weights).sum().backward()

    for name, got, want in (("d_symm", ds, wds), ("d_asymm", da, wda), ("mos", mos, wmos),
                            ("loss", loss, wloss)):
        got, want = got.detach().double().cpu(), want.detach()
        assert float(((got - want).abs() / want.abs()).max()) < 1e-5, name
    for name, got, want in (("g_ref", g_ref, rd.grad), ("g_deg", g_deg, dd.grad)):
        err = float((got.double().cpu() - want).abs().max() / want.abs().max())
        assert err < 2e-5, (name, err)


def test_other_geometry_rejects_too_few_frames():
    from torch_pesq import PesqLossTriton

    model = PesqLossTriton(0.5, sample_rate=16000, n_fft=256, win_length=256, hop_length=512).cuda()
    x = torch.randn(1, 8000, device="cuda")
    with pytest.raises(ValueError, match="20 frames"):
        model(x, x)


@pytest.mark.parametrize("n_fft, hop", [(512, 160), (512, 512), (1024, 256), (1024, 1024), (256, 64)])
@pytest.mark.parametrize("rows, nsamples", [(1, 1024), (3, 1025), (2, 4099), (40, 70001)])
def test_transforms_at_odd_frame_counts(n_fft, hop, rows, nsamples):
    """The radix-4, radix-8 and radix-2 transforms with one to four frames per
    wavefront (chosen by the grid), last wavefronts partly filled, rows at odd
    offsets: a row equals the same row alone bit for bit, and the float64
    operator within the module's budgets (forward 1e-5 relative + 5e-6 of the
    frame, backward + 1e-5 of the sample scale)."""

    mod, window, scale = _module(n_fft, 49, hop)
    signal = 1000.0 * torch.randn(rows, nsamples, generator=torch.Generator().manual_seed(nsamples))
    got, want, g_got, g_want = _both(mod, window, scale, signal.cuda())
    assert _violation(got, want, ATOL_FWD, _frame_scale(want)) <= 0.0
    assert _violation(g_got, g_want, ATOL_BWD, _sample_scale(g_want, hop, mod.novertaps)) <= 0.0
    x = signal.cuda().requires_grad_(True)
    y = mod(x)
    (g,) = torch.autograd.grad(y.sum(), x)
    x1 = signal[-1:].cuda().requires_grad_(True)
    y1 = mod(x1)
    (g1,) = torch.autograd.grad(y1.sum(), x1)
    assert torch.equal(y[-1:], y1) and torch.equal(g[-1:], g1)


@pytest.mark.parametrize("n_fft, win_length, hop", [(64, 64, 37), (256, 200, 64), (512, 400, 160), (1024, 1024, 300)])
@pytest.mark.parametrize("rate, nsamples", [(16000, 12001), (8000, 9003), (44100, 36007)])
def test_loss_runs_the_operators_composed(n_fft, win_length, hop, rate, nsamples):
    """The whole loss against its stand-alone operators in the reference's order
    (common peak first), each input alone and both requiring a gradient, over
    odd lengths, hops that leave ragged frames, and batches whose tiles pass
    through the band totals (more than 64).  Both hold the transforms and
    recursions in float64 and store each stage in float32: values within 2e-6
    relative; gradients within 1e-4 of the row's peak, for a frame whose
    disturbance lies at its dead zone takes either side."""

    from bench import speech_like_pair
    from torch_pesq import PesqLossTriton
    from torch_pesq.hip_ops.elementwise import peak_normalize, pesq_epilogue

    model = PesqLossTriton(0.5, sample_rate=rate, n_fft=n_fft, win_length=win_length,
                           hop_length=hop).cuda()
    ref, deg = speech_like_pair(3, nsamples, seed=n_fft, noise=0.1)
    signals = [torch.from_numpy(x).cuda() for x in (ref, deg)]

    def composed(r, d):
        x = model.resampler(peak_normalize(r, d, stack=True)) if rate != 16000 else peak_normalize(r, d, stack=True)
        y = model.preemphasize(model.align_level(x))
        n = x.shape[1]
        spectral = HipStftBark(model.to_spec.window, model.fbank.fbank,
                               model.fbank.pow_dens_correction, n_fft, hop).cuda()
        bark = spectral(y, n + n % 256)
        ds, da = model.chain(bark[:3], bark[3:])
        mos, loss = pesq_epilogue(ds, da, 0.5)
        return ds, da, mos, loss

    for need in ((True, True), (True, False), (False, True), (False, False)):
        runs = []
        for f in (model._run, composed):
            ins = [x.clone().requires_grad_(n) for x, n in zip(signals, need)]
            out = f(*ins)
            want = [x for x in ins if x.requires_grad]
            grads = torch.autograd.grad(out[2].sum() + out[3].sum(), want) if want else ()
            runs.append((out, grads))
        (got, g_got), (want, g_want) = runs
        for a, b in zip(got, want):
            torch.testing.assert_close(a.detach(), b.detach(), rtol=2e-6, atol=0.0)
        for a, b in zip(g_got, g_want):
            assert float(((a - b).abs().amax(1) / b.abs().amax(1)).max()) < 1e-4


@pytest.mark.parametrize("bad", [float("inf"), -float("inf"), float("nan")])
def test_general_loss_at_infinities(bad):
    """An infinite sample is the common peak: neither signal of its pair keeps a
    gradient; a NaN is not, and the other signal keeps its own.  Other pairs
    are untouched."""

    from torch_pesq import PesqLossTriton

    model = PesqLossTriton(0.5, sample_rate=16000, hop_length=160).cuda()
    x = torch.randn(2, 2, 9001, generator=torch.Generator().manual_seed(1)).cuda()
    want = model(x[0], x[1])
    y = x.clone()
    y[0, 0, 777] = bad
    r, d = y[0].requires_grad_(True), y[1].requires_grad_(True)
    loss = model(r, d)
    g_ref, g_deg = torch.autograd.grad(loss.sum(), [r, d])
    assert loss[1] == want[1]
    assert not g_ref[0].isfinite().any() and g_ref[1].isfinite().all()
    assert g_deg[0].isfinite().all() == (bad != bad) and g_deg[1].isfinite().all()


@pytest.mark.parametrize("n_fft, win_length, hop", [(512, 400, 160), (1024, 1024, 256)])
@pytest.mark.parametrize("rate, nsamples", [(16000, 12001), (8000, 9003), (44100, 36007)])
def test_general_loss_over_the_whole_float32_range(rate, nsamples, n_fft, win_length, hop):
    """The loss does not depend on the signals' scale: times a power of two it has
    the same bits, the gradients times its inverse, also where the samples are
    subnormal (the smallest are 2^-142 here) and where the peak is next to the
    largest float32."""

    from torch_pesq import PesqLossTriton

    model = PesqLossTriton(0.5, sample_rate=rate, n_fft=n_fft, win_length=win_length,
                           hop_length=hop).cuda()
    x = torch.randn(2, 3, nsamples, generator=torch.Generator().manual_seed(7)) * 0.2
    x[1] = x[0] + 0.3 * x[1]
    x = ((x.clamp(-0.999, 0.999) * 4096).round() / 4096).double()  # exact at every scale below
    x[0, :, 100] = 0.999755859375  # 4095 / 4096, the common peak

    def run(power):
        y = (x * 2.0 ** power).float().cuda()
        assert torch.equal(y.cpu().double(), x * 2.0 ** power)
        r, d = y[0].requires_grad_(True), y[1].requires_grad_(True)
        loss = model(r, d)
        return (loss.detach(),) + torch.autograd.grad(loss.sum(), [r, d])

    loss, g_ref, g_deg = run(0)
    assert loss.isfinite().all() and g_ref.isfinite().all() and g_deg.isfinite().all()
    for power in (-130, -100, -13, 20, 100, 128):
        got, got_ref, got_deg = run(power)
        assert torch.equal(got, loss), power
        for got_g, want_g in ((got_ref, g_ref), (got_deg, g_deg)):
            exact = want_g.double() * 2.0 ** -power
            # (subnormal ones: from the float64 value, not from its float32 rounding)
            close = (exact.abs() < 2.0 ** -126) & ((got_g.double() - exact).abs() < 2.0 ** -149)
            assert bool(((got_g == exact.float()) | close).all()), power


@pytest.mark.parametrize("rate", [16000, 44100])
def test_general_loss_create_graph_and_double_backward(rate):
    """``create_graph`` gives the same first derivatives (the signals' common
    factor is then applied by torch's operators), the second ones raise."""

    from torch_pesq import PesqLossTriton

    model = PesqLossTriton(0.5, sample_rate=rate, hop_length=160).cuda()
    x = torch.randn(2, 2, rate, generator=torch.Generator().manual_seed(3)) * 0.05
    ref, deg = x[0].cuda().requires_grad_(True), x[1].cuda().requires_grad_(True)
    want = torch.autograd.grad(model(ref, deg).sum(), [ref, deg])
    got = torch.autograd.grad(model(ref, deg).sum(), [ref, deg], create_graph=True)
    assert all(torch.equal(g, w) and not g.requires_grad for g, w in zip(got, want))
    upstream = torch.ones(2, device="cuda", requires_grad=True)
    got = torch.autograd.grad(model(ref, deg), [ref, deg], grad_outputs=upstream, create_graph=True)
    assert all(torch.equal(g, w) and g.requires_grad for g, w in zip(got, want))
    with pytest.raises(RuntimeError, match="differentiate twice"):
        (got[0].sum() + got[1].sum()).backward()
    # one signal's gradient alone, and one output's
    d_symm, d_asymm = model.raw(ref.detach(), deg)
    (g1,) = torch.autograd.grad(d_symm.sum(), deg)
    d_symm, _ = model.raw(ref, deg.detach())
    (g2,) = torch.autograd.grad(d_symm.sum(), ref)
    d_symm, _ = model.raw(ref, deg)
    both = torch.autograd.grad(d_symm.sum(), [ref, deg])
    assert torch.equal(g1, both[1]) and torch.equal(g2, both[0])


@pytest.mark.parametrize("batch, nsamples", [(700, 6145), (37, 116961)])
def test_general_loss_of_large_grids_scales_every_pair(batch, nsamples):
    """Grids whose scans run segments (rows of one and of several): pairs at any
    scale among the others give what they give alone, by the lane-state scans
    (float64 either way, rounded to float32 rows: 1e-6 of the gradient's peak)."""

    from torch_pesq import PesqLossTriton

    assert 2 * batch * -(-nsamples // 1024) > 8192
    model = PesqLossTriton(0.5, sample_rate=16000, hop_length=160).cuda()
    gen = torch.Generator(device="cuda").manual_seed(nsamples)
    x = torch.randn(2, batch, nsamples, generator=gen, device="cuda") * 0.05
    x[1] = x[0] + 0.4 * x[1]
    power = torch.zeros(batch, device="cuda", dtype=torch.float64)
    power[1], power[batch // 2], power[-2] = -110.0, 100.0, 30.0
    y = (x.double() * torch.exp2(power)[:, None]).float()

    def run(z):
        r, d = z[0].contiguous().requires_grad_(True), z[1].contiguous().requires_grad_(True)
        loss = model(r, d)
        return (loss.detach(),) + torch.autograd.grad(loss.sum(), [r, d])

    loss, *grads = run(y)
    for first in (0, batch // 2, batch - 3):
        item = slice(first, first + 3)
        want_loss, *want = run(x[:, item])
        assert float(((loss[item] - want_loss).abs() / want_loss).max()) < 1e-6
        for got, w in zip(grads, want):
            got = got[item].double() * torch.exp2(power[item])[:, None]
            peak = w.abs().amax(1, keepdim=True)
            assert float(((got - w).abs() / peak).max()) < 1e-6
