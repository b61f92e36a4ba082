"""The 3D kernel for separable element grids (rows of the aperture in
registers) and the general 3D kernel, bit for bit against the FP32 oracle at
the sizes and on the sides of the rule where they can go wrong: batches of
four rows cut short, one row or column, more rows or columns than a pass, an
array that is not a grid, offsets and delays out of range, fewer channels
than elements, float RF with values that are not finite."""
import numpy as np
import pytest

from dataclasses import replace

from oracle import oracle as O
from supra_amd import workloads as W
from supra_amd.beamformer import RxBeamformer, USRawData

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


def volume(lx, ly, n_lines, n_depths, n_samples, channels=None):
    w = W.matrix_3d_small(n_el=max(lx, ly), n_lines=n_lines, n_depths=n_depths, n_samples=n_samples)
    bf = replace(w.bf, element_layout=(lx, ly), max_aperture=(lx, ly), tx_max_aperture=(lx, ly))
    return replace(w, bf=bf, num_channels=channels or lx * ly)


def both(w, g, rf, **over):
    kw = dict(w.das_kwargs(), **over)
    eng = RxBeamformer(g)
    img = eng.perform_rx_beamforming(0, USRawData(torch.from_numpy(rf).cuda(), w.fs_hz, g), kw["f_number"],
                                     kw["speed_of_sound_mm_per_s"], kw["window_type"], kw["window_parameter"],
                                     kw["interpolate_transmits"], kw["additional_offset"])
    torch.cuda.synchronize()
    out = img.data.cpu().numpy()
    eng.close()
    return out, O.das(g, rf, w.fs_hz, **kw)


def assert_same(gpu, ref):
    same = (gpu == ref) | (np.isnan(gpu) & np.isnan(ref))
    assert same.all(), f"{(~same).sum()} of {gpu.size} voxels differ, first {np.argwhere(~same)[0]}"


@pytest.mark.parametrize("lx,ly,n_depths,n_samples,channels", [
    (2, 2, 70, 300, None), (9, 3, 130, 500, None), (5, 7, 257, 500, None), (4, 33, 90, 400, None),
    (33, 4, 90, 400, None), (40, 6, 64, 300, None), (6, 40, 64, 300, None), (8, 8, 150, 700, 24)])
def test_row_and_column_edges(device, lx, ly, n_depths, n_samples, channels):
    rng = np.random.default_rng(lx * 100 + ly)
    w = volume(lx, ly, 5, n_depths, n_samples, channels)
    rf = rng.integers(-20000, 20000, w.rf_shape).astype(np.int16)
    assert_same(*both(w, w.geometry(), rf))


@pytest.mark.parametrize("f_number,offset", [(0.5, 0), (4.0, 0), (1.0, 5), (1.0, -60), (1.0, 400)])
def test_apertures_and_offsets(device, f_number, offset):
    """Mostly far field, mostly near field, and delays that leave the RF at
    either end (with no offset the deepest voxels leave it)."""
    w = volume(8, 8, 4, 200, 300)
    rf = np.random.default_rng(1).integers(-20000, 20000, w.rf_shape).astype(np.int16)
    assert_same(*both(w, w.geometry(), rf, f_number=f_number, additional_offset=offset))


@pytest.mark.parametrize("axis", [0, 1])
def test_array_off_the_grid(device, axis):
    """One moved element: the general kernel."""
    w = volume(6, 6, 4, 150, 500)
    g = replace(w.geometry())
    pos = (g.element_x if axis == 0 else g.element_y).copy()
    pos[14] += 0.05
    g = replace(g, **({"element_x": pos} if axis == 0 else {"element_y": pos}))
    rf = np.random.default_rng(2).integers(-20000, 20000, w.rf_shape).astype(np.int16)
    assert_same(*both(w, g, rf))


def test_float_rf_with_infinities(device):
    """An infinite or NaN sample reaches exactly the voxels it reaches in the
    reference: an element outside the aperture or out of range adds nothing."""
    w = volume(7, 5, 4, 200, 300)
    rng = np.random.default_rng(3)
    rf = rng.normal(size=w.rf_shape).astype(np.float32) * 100
    rf[3, 4, 250:] = np.inf
    rf[5, :, 120] = np.nan
    rf[7, 20, 299] = -np.inf
    assert_same(*both(w, w.geometry(), rf))
