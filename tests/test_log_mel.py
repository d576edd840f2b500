"""The log-mel launch at its edges (csrc/kernels/audio.hip): frame counts that are no multiple
of a workgroup's, both band counts, time-major rows with padding columns, and the encoder on
them for 80 bands."""
import numpy as np
import pytest
import torch

from loqa_hub_amd import ops
from loqa_hub_amd.ops import reference as ref


def test_band_ranges_hold_every_weight():
    for n in (80, 128):
        c = ref.MelConstants.create(n)
        j = torch.arange(201)
        inside = (j >= c.ranges[:, :1]) & (j < c.ranges[:, 1:])
        assert (c.filters[~inside] == 0).all() and (c.filters.sum(1) > 0).all()
        odd = ref.MelConstants(2, c.window, c.cos_basis, c.sin_basis, torch.zeros(2, 201))
        assert (odd.ranges == 0).all()


@pytest.mark.gpu
@pytest.mark.parametrize("n_mels", [80, 128])
@pytest.mark.parametrize("samples", [201, 1600, 2560, 16000 * 3 + 77])
def test_rows_against_float64(n_mels, samples):
    c = ref.MelConstants.create(n_mels)
    x = torch.from_numpy(0.1 * np.random.RandomState(samples).randn(3, samples)).float()
    x[1] *= 1e-3
    x[2, samples // 2:] = 0
    frames = samples // 160
    st = torch.stft(x.double(), 400, 160, window=c.window.double(), return_complex=True, center=True, pad_mode="reflect")
    lg = (c.filters.double() @ st[..., :frames].abs().square()).clamp(min=1e-10).log10()
    want = (torch.maximum(lg, lg.amax((1, 2), keepdim=True) - 8) + 4) / 4
    got = ops.log_mel(x.cuda(), c).cpu()
    rows = ops.log_mel_rows(x.cuda(), c, 192).cpu().view(3, frames, 192)
    # bf16 (values of a few units: half an ulp of up to 2^-8); f32 power sums before the logarithm
    assert (got.double() - want).abs().max() <= 2.0 ** -8 * want.abs().clamp(min=1).max() + 1e-3
    assert torch.equal(rows[..., :n_mels].transpose(1, 2), got) and (rows[..., n_mels:] == 0).all()


@pytest.mark.gpu
@pytest.mark.parametrize("B,samples", [(1, 16 * 160 * 256), (1, 16 * 160 * 256 + 160), (7, 48 * 2560 + 800), (300, 400)])
def test_workgroups_that_take_several_groups_of_frames(B, samples):
    c = ref.MelConstants.create(80)
    x = torch.from_numpy(0.1 * np.random.RandomState(samples).randn(B, samples)).float()
    x *= torch.logspace(0, -2, B)[:, None]                # utterances of different maxima
    frames = samples // 160
    st = torch.stft(x.double(), 400, 160, window=c.window.double(), return_complex=True, center=True, pad_mode="reflect")
    lg = (c.filters.double() @ st[..., :frames].abs().square()).clamp(min=1e-10).log10()
    want = ((torch.maximum(lg, lg.amax((1, 2), keepdim=True) - 8) + 4) / 4).transpose(1, 2)
    for cols in (192, 83):                                # four columns a lane, and rows that are not aligned
        rows = ops.log_mel_rows(x.cuda(), c, cols).cpu().view(B, frames, cols)
        # the bound of the test above
        assert (rows[..., :80].double() - want).abs().max() <= 2.0 ** -8 * want.abs().clamp(min=1).max() + 1e-3
        assert (rows[..., 80:] == 0).all()


@pytest.mark.gpu
def test_encoder_of_80_bands_on_the_tiled_path(monkeypatch):
    from loqa_hub_amd.models import whisper as wm
    from loqa_hub_amd.models.configs import whisper_config
    w = wm.WhisperWeights(whisper_config("test-whisper", enc_layers=3), torch.device("cuda", 0), seed=3)
    model = wm.WhisperModel(w)
    audio = (torch.rand(2, 480000, device="cuda", generator=torch.Generator("cuda").manual_seed(5)) - 0.5) * 0.2
    a = model.encode(audio).float()
    monkeypatch.setattr(wm, "ENC_TILE", False)
    b = model.encode(audio).float()
    # the two paths round the residual stream at other places: a few bf16 ulps after three layers
    assert (a - b).norm() <= 0.01 * b.norm()


@pytest.mark.gpu
@pytest.mark.parametrize("value", [float("inf"), float("-inf"), float("nan")])
def test_samples_that_are_not_finite_cost_their_frames_only(value):
    c = ref.MelConstants.create(80)
    x = torch.from_numpy(0.1 * np.random.RandomState(3).randn(2, 16000)).float()
    bad = x.clone()
    bad[0, 8000] = value
    st = torch.stft(x.double(), 400, 160, window=c.window.double(), return_complex=True, center=True, pad_mode="reflect")
    lg = (c.filters.double() @ st[..., :100].abs().square()).clamp(min=1e-10).log10()
    lg[0, :, 49:52] = -10                                 # 160 t - 200 <= 8000 < 160 t + 200: silence
    want = (torch.maximum(lg, lg.amax((1, 2), keepdim=True) - 8) + 4) / 4
    got = ops.log_mel(bad.cuda(), c).cpu()
    assert (got.double() - want).abs().max() <= 2.0 ** -8 * want.abs().clamp(min=1).max() + 1e-3
