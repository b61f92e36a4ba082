"""Minimum variance of well-loaded systems (csrc/mv_block.hip) at the edges of
its blocks, sub-blocks and tiles, and the rule that chooses between it and the
kernel that refines weakly loaded systems, against the FP64 oracle."""
import numpy as np
import pytest

from oracle import oracle as O
from supra_amd.beamformer import USRawData, mv_perform_rx_beamforming

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


def gpu_mv(x, *args, **kw):
    img = mv_perform_rx_beamforming(USRawData(torch.from_numpy(np.ascontiguousarray(x)).cuda(), 1.0, None, 1, (1, 1)),
                                    *args, **kw)
    torch.cuda.synchronize()
    return img.data.cpu().numpy()


def apertures(rng, n_rx, n_ch, n_d, dtype=np.float32):
    """Random apertures, some shorter than any sub-array, one sample empty."""
    x = (rng.normal(size=(n_rx, n_ch, n_d)) * 100).astype(dtype)
    f = rng.integers(0, max(1, n_ch // 3), (n_rx, n_d))
    last = np.minimum(n_ch - 1, f + rng.integers(0, n_ch, (n_rx, n_d)))
    ch = np.arange(n_ch)[None, :, None]
    x[(ch < f[:, None, :]) | (ch > last[:, None, :])] = 0
    x[:, :, n_d // 2] = 0
    return x


def check(gpu, ref, L, alpha):
    # FP32 factorisation of a system of condition number at most 1 + L / alpha:
    # a few units of 2^-24 times it, relative to the system's own scale; the
    # outputs are compared relative to the larger of themselves and 1e-3 of
    # the image's peak, since an output may cancel
    err = np.abs(gpu.astype(np.float64) - ref) / np.maximum(np.abs(ref), 1e-3 * np.abs(ref).max())
    kappa = 1.0 + L / alpha
    assert np.quantile(err, 0.99) < max(1e-5, 16 * kappa * 2.0**-24), np.quantile(err, 0.99)
    assert err.max() < max(1e-4, 1000 * kappa * 2.0**-24), err.max()


@pytest.mark.parametrize("L,T,n_ch,n_d,means", [
    (1, 0, 5, 7, False), (15, 1, 40, 33, False), (16, 5, 32, 70, True), (17, 5, 40, 70, False), (31, 3, 64, 45, True),
    (32, 0, 64, 25, False), (32, 8, 70, 60, False), (33, 5, 70, 40, True), (48, 2, 96, 31, False),
    (49, 7, 128, 23, False), (64, 5, 65, 36, False), (64, 10, 256, 24, True), (64, 32, 128, 40, False)])
def test_block_edges(device, L, T, n_ch, n_d, means):
    """Sub-array sizes on both sides of every block edge, windows shorter and
    longer than a tile, tiles cut by the last sample, with and without means."""
    x = apertures(np.random.default_rng(L * 100 + T), 3, n_ch, n_d)
    gpu = gpu_mv(x, L, T, 1.5, means, 0.1)
    check(gpu, O.mv(x, L, T, 1.5, means, 0.1), L, 0.1)
    assert (gpu[n_d // 2] == 0).all() == (O.mv(x, L, T, 1.5, means, 0.1)[n_d // 2] == 0).all()


@pytest.mark.parametrize("L", [16, 32, 64])
def test_both_sides_of_the_loading_rule(device, L):
    """1 + L / alpha just below and above the bound of the refined kernel:
    both sides meet the FP64 oracle and each other."""
    x = apertures(np.random.default_rng(L), 2, 2 * L, 50, np.int16)
    lo, hi = L / 10050.0, L / 9950.0
    a, b = gpu_mv(x, L, 4, 1.5, False, lo), gpu_mv(x, L, 4, 1.5, False, hi)
    check(a, O.mv(x, L, 4, 1.5, False, lo), L, lo)
    check(b, O.mv(x, L, 4, 1.5, False, hi), L, hi)


@pytest.mark.parametrize("L,T,value", [(16, 3, np.inf), (32, 5, np.nan), (32, 5, -3.4e38), (64, 2, 1e20)])
def test_samples_without_a_finite_covariance(device, L, T, value):
    """Every window that holds such a sample is 0, every other output keeps
    its bits."""
    rng = np.random.default_rng(3)
    x = rng.normal(size=(2, 2 * L, 60)).astype(np.float32)
    clean = gpu_mv(x, L, T, 1.5, False, 0.1)
    x[1, L, 31] = value
    got = gpu_mv(x, L, T, 1.5, False, 0.1)
    hit = np.zeros_like(clean, dtype=bool)
    hit[31 - T:31 + T + 1, 1] = True
    assert (got[hit] == 0).all() and (clean[hit] != 0).all()
    assert np.array_equal(got[~hit], clean[~hit])


def test_weak_windows_next_to_a_strong_echo(device):
    """Windows of unit samples on either side of one 1e9 times as strong keep
    their own precision: no window sum is formed by subtraction."""
    rng = np.random.default_rng(8)
    x = rng.normal(size=(1, 64, 64)).astype(np.float32)
    x[:, :, 30] *= 1e9
    T = 3
    gpu, ref = gpu_mv(x, 32, T, 1.5, False, 0.1)[:, 0], O.mv(x, 32, T, 1.5, False, 0.1)[:, 0]
    far = np.abs(np.arange(64) - 30) > T
    check(gpu[far], ref[far], 32, 0.1)
