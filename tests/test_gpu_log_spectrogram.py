"""The one-pass log power spectrogram against torch.stft in float64 (clips shorter
than a frame, lengths inside and at the edges of a hop, mono and stereo in one
batch, non-finite samples past a length), and the eight-channel band means
against the general kernel."""

import pytest
import torch

from trifusion_amd.kernels.block import bands, log_spectrogram

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("n,c", [(1, 1), (159, 2), (160, 1), (401, 2), (8000, 1), (64000, 2)])
def test_against_float64(n, c):
    g = torch.Generator().manual_seed(n + c)
    audio = torch.randn(4, c, n, generator=g) * torch.tensor([1.0, 0.1, 1e-3, 3.0])[:, None, None]
    lengths = torch.tensor([n, max(n - 1, 0), n // 2, 0])
    channels = torch.tensor([c, 1, c, 1])
    keep = (torch.arange(n) < lengths[:, None])[:, None] & (torch.arange(c) < channels[:, None])[..., None]
    wave = audio.masked_fill(~keep, 0)
    window = torch.hann_window(400, periodic=True)
    # what lies past a length is never read
    y = log_spectrogram(torch.where(keep, audio, torch.nan).to(DEV), window.to(DEV), lengths.to(DEV),
                        channels.to(DEV)).cpu()
    spec = torch.stft(wave.double().reshape(4 * c, n), n_fft=512, hop_length=160, win_length=400,
                      window=window.double(), center=True, pad_mode="constant", return_complex=True)
    mag = spec.abs().reshape(4, c, 257, -1)
    power = mag.square().sum(1) / channels[:, None, None]
    frames = n // 160 + 1
    valid = (torch.arange(frames) < (lengths // 160 + 1)[:, None])[..., None]
    assert y.shape == (4, frames, 257) and not y.masked_fill(valid, 0).any()
    got = (y.double().exp() - 1e-6).transpose(1, 2)
    # nine butterfly levels, each within 2^-23 of the frame's norm (||X|| = sqrt(512) ||x||),
    # and the fp32 logarithm (values up to ~15) with its argument's rounding
    norm = (mag.square().sum(2, keepdim=True)).sqrt().amax(1)
    delta = 9 * 2.0**-23 * norm
    bound = 2 * mag.amax(1) * delta + delta**2 + (power + 1e-6) * 20 * 2.0**-23
    err = ((got - power).abs() - bound * c).masked_fill(~valid.transpose(1, 2), -1)
    assert err.max() <= 0, err.max()


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("b,t,f,c", [(1, 1, 8, 8), (2, 5, 65, 64), (1, 3, 33, 128), (2, 2, 9, 24)])
def test_bands_by_pieces(b, t, f, c, dtype):
    x = torch.randn(b, t, f, c, generator=torch.Generator().manual_seed(f)).to(dtype).to(DEV)
    y = bands(x.permute(0, 3, 1, 2))  # channels last: pieces of eight
    assert torch.equal(y, bands(x.permute(0, 3, 1, 2).contiguous()))


def test_short_lengths_are_refused():
    audio, window = torch.zeros(4, 1, 400, device=DEV), torch.ones(400, device=DEV)
    whole, short = torch.full((4,), 400, device=DEV), torch.full((3,), 1, device=DEV)
    for lengths, channels in ((short, whole), (whole, short)):
        with pytest.raises(ValueError, match="entry per clip"):
            log_spectrogram(audio, window, lengths, channels)
