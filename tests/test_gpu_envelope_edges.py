"""Envelope kernel at the edges of its groups of taps, its row tiles and the
route that sums every tap, bit for bit against the FP32 oracle."""
import numpy as np
import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


def gpu_envelope(img, n_taps):
    from supra_amd.postprocess import HilbertFirEnvelope
    env = HilbertFirEnvelope(n_taps).demodulate(torch.from_numpy(img).cuda(), torch.float32)
    torch.cuda.synchronize()
    return env.data.cpu().numpy()


def check(img, n_taps):
    got = gpu_envelope(img, n_taps)
    frames = img[None] if img.ndim == 2 else img
    ref = np.stack([O.clamp_cast(O.envelope(f, n_taps), np.float32) for f in frames]).reshape(img.shape)
    assert np.array_equal(got, ref), f"{(got != ref).sum()} of {got.size} samples differ"


@pytest.mark.parametrize("n_taps", [1, 2, 3, 4, 15, 16, 17, 18, 32, 33, 34, 35, 129, 256])
def test_tap_counts(device, n_taps):
    rng = np.random.default_rng(n_taps)
    check((rng.normal(size=(83, 66)) * 1000).astype(np.float32), n_taps)


@pytest.mark.parametrize("shape", [(1, 1), (31, 64), (32, 65), (33, 63), (64, 1), (65, 130), (9, 64, 64), (9, 65, 64),
                                   (520, 3, 2), (256, 65, 65)])
def test_row_tiles(device, shape):
    """Images around both tile heights; the last two launch enough workgroups
    for the tall tiles."""
    rng = np.random.default_rng(sum(shape))
    check((rng.normal(size=shape) * 1000).astype(np.float32), 33)


@pytest.mark.parametrize("value", [np.inf, -np.inf, np.nan, 3.0e38, 1.0e-30])
def test_extreme_samples(device, value):
    """Infinities and NaN reach every window that holds them (0 times them is
    NaN), overflowing and underflowing squares as in the reference."""
    rng = np.random.default_rng(5)
    img = rng.normal(size=(200, 70)).astype(np.float32)
    img[77, 3] = value
    img[130:, 40] = value
    img[:, 60] = 0.0
    check(img, 65)


@pytest.mark.parametrize("n_taps", [1, 2, 3])
@pytest.mark.parametrize("shape", [(520, 3, 2), (256, 65, 65)])
def test_short_filters_of_many_frames(device, n_taps, shape):
    """Filters that sum every tap keep short tiles without padding rows, also
    where the other filters take the tall ones."""
    rng = np.random.default_rng(n_taps)
    img = (rng.normal(size=shape) * 1000).astype(np.float32)
    img[1, -1, 0], img[-1, 0, -1] = np.nan, np.inf
    check(img, n_taps)
