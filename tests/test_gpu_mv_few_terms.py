"""Minimum variance of windows that hold few sub-array vectors (the system in
the space of the terms, csrc/mv_block.hip) against the FP64 oracle: apertures
around the sub-array length, so that the number of terms crosses its limit of
15 in neighbouring tiles, smoothing lengths up to the limit, samples that are
all zero or not finite, and weak loadings."""
import numpy as np
import pytest

from oracle import oracle as O
from supra_amd.beamformer import USRawData, mv_perform_rx_beamforming

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


def gpu_mv(x, *args):
    img = mv_perform_rx_beamforming(USRawData(torch.from_numpy(np.ascontiguousarray(x)).cuda(), 1.0, None, 1, (1, 1)), *args)
    torch.cuda.synchronize()
    return img.data.cpu().numpy()


def signals(rng, n_rx, n_ch, n_d, lengths, dtype=np.float32):
    """Random apertures of the given lengths (cycled over depth)."""
    x = (rng.normal(size=(n_rx, n_ch, n_d)) * 200).astype(dtype)
    ch = np.arange(n_ch)
    for s in range(n_rx):
        for d in range(n_d):
            ln = min(n_ch, lengths[(d + 3 * s) % len(lengths)])
            f = int(rng.integers(0, n_ch - ln + 1))
            x[s, (ch < f) | (ch >= f + ln), d] = 0
    return x


# FP64 up to the two numbers the output is formed from: their rounding, powf
# and the division, ~8 units of 2^-24, relative to the larger of the output
# and 1e-3 of the peak (an output may cancel).  Tiles with more terms factorise
# in FP32: 1000 kappa 2^-24 for the worst output.
def check(gpu, ref, L, alpha, few):
    err = np.abs(gpu.astype(np.float64) - ref) / np.maximum(np.abs(ref), 1e-3 * np.abs(ref).max())
    assert err.max() < (5e-6 if few else max(1e-4, 1000 * (1.0 + L / alpha) * 2.0**-24)), err.max()


@pytest.mark.parametrize("L,T,n_ch,n_d,alpha", [
    (2, 5, 9, 40, 0.1), (16, 7, 40, 33, 0.1), (17, 0, 64, 50, 0.02), (32, 5, 64, 61, 0.01), (33, 6, 70, 29, 0.1),
    (48, 1, 128, 35, 0.1), (64, 5, 128, 50, 0.01), (64, 7, 100, 17, 1.0)])
def test_one_sub_array_per_sample(device, L, T, n_ch, n_d, alpha):
    """Apertures no longer than the sub-array: 2T + 1 terms, fewer at the ends."""
    x = signals(np.random.default_rng(L + T), 3, n_ch, n_d, [L, L - 1, max(1, L // 2), L, 1])
    x[0, :, n_d // 3:n_d // 3 + 2] = 0
    check(gpu_mv(x, L, T, 1.5, False, alpha), O.mv(x, L, T, 1.5, False, alpha), L, alpha, True)


@pytest.mark.parametrize("L,T,dtype", [(16, 2, np.int16), (32, 3, np.float32), (64, 1, np.int16), (64, 4, np.float32)])
def test_terms_on_both_sides_of_the_limit(device, L, T, dtype):
    """Depth ranges with one, two and many sub-arrays per sample."""
    rng = np.random.default_rng(L * T)
    x = np.concatenate([signals(rng, 2, 2 * L, n, ln, dtype) for n, ln in
                        ((30, [L]), (25, [L, L + 1]), (25, [L + 2]), (20, [L, 2 * L]), (30, [L - 1, L]))], axis=2)
    check(gpu_mv(x, L, T, 1.5, False, 0.1), O.mv(x, L, T, 1.5, False, 0.1), L, 0.1, False)


@pytest.mark.parametrize("value", [np.inf, np.nan, 1e20])
def test_not_finite_samples_leave_the_others(device, value):
    """Windows with such a sample are 0, every other output keeps its bits."""
    L, T = 32, 5
    x = signals(np.random.default_rng(1), 2, 48, 70, [L])
    clean = gpu_mv(x, L, T, 1.5, False, 0.1)
    c = np.nonzero(x[1, :, 40])[0][L // 2]
    x[1, c, 40] = value
    got = gpu_mv(x, L, T, 1.5, False, 0.1)
    hit = np.zeros_like(clean, dtype=bool)
    hit[40 - T:40 + T + 1, 1] = True
    assert (got[hit] == 0).all() and np.array_equal(got[~hit], clean[~hit])
