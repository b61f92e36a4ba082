"""F-numbers so small that the aperture of the deeper pixels is infinite in
single precision: every element of a transmit's aperture is in it and no other,
in the 3D kernel that pads its rows to four (bit for bit the FP32 oracle) and in
the adjoint, whose waves take two elements each."""
from dataclasses import replace

import numpy as np
import pytest

from oracle import oracle as O
from supra_amd import _native as N
from supra_amd import workloads as W
from supra_amd.beamformer import RxBeamformer, USRawData

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")

TINY = 2e-38


@pytest.mark.parametrize("dtype", [np.int16, np.float32])
@pytest.mark.parametrize("lx,ly", [(4, 5), (6, 31)])
def test_das_3d(device, dtype, lx, ly):
    w = W.matrix_3d_small(n_el=max(lx, ly), n_lines=4, n_depths=130, n_samples=1300)
    w = replace(w, bf=replace(w.bf, element_layout=(lx, ly), max_aperture=(lx, ly), tx_max_aperture=(lx, ly)),
                num_channels=lx * ly)
    g = w.geometry()
    rf = np.random.default_rng(ly).integers(-20000, 20000, w.rf_shape).astype(dtype)
    kw = dict(w.das_kwargs(), f_number=TINY)
    eng = RxBeamformer(g)
    img = eng.perform_rx_beamforming(N.BF_DELAY_AND_SUM, USRawData(torch.from_numpy(rf).cuda(), w.fs_hz, g), TINY,
                                     kw["speed_of_sound_mm_per_s"], kw["window_type"], 0.0, False, 0)
    torch.cuda.synchronize()
    ref = O.das(g, rf, w.fs_hz, **kw)
    assert (ref != 0).any()
    assert np.array_equal(img.data.cpu().numpy(), ref)
    eng.close()


@pytest.mark.parametrize("elements,shared", [(9, False), (11, True)])
def test_adjoint(device, elements, shared):
    """Odd apertures leave half a wave's pair past the last element; with
    several writers per line such an element would add to channel 0."""
    from supra_amd.differentiable import DifferentiableDAS
    w = W.linear_2d(num_scatterers=1)
    w = replace(w, bf=replace(w.bf, element_layout=(elements, 1), num_scanlines=(4, 1), max_aperture=(elements, 1),
                              tx_max_aperture=(elements, 1), num_depths=150), num_channels=elements, num_samples=2300)
    g = w.geometry()
    scan = g.scanlines.copy()
    scan["tx"]["last"][..., 0] = elements - 2
    g = replace(g, scanlines=scan)
    assert elements % 2 == 1 and (scan["tx"]["first"][..., 0] == 0).all()
    channels = elements
    if shared:
        channels = (elements + 1) // 2
        g = replace(g, element_to_channel=(np.arange(elements) % channels).astype(np.int32))
    rng = np.random.default_rng(elements)
    rf = rng.normal(size=(1, 4, channels, 2300)).astype(np.float32)
    gi = rng.normal(size=(1, 150, 4)).astype(np.float32)
    c_mm = np.array([1540.0e3])
    dd = DifferentiableDAS(g, w.fs_hz, TINY, N.WINDOW_HAMMING)
    x, c = torch.from_numpy(rf).cuda(), torch.tensor(c_mm / 1000.0, dtype=torch.float64, device="cuda")
    _, norm = dd.forward_raw(x, c)
    grad_rf, grad_c = dd.adjoint_raw(x, c, norm, torch.from_numpy(gi).cuda())
    got_rf, got_c = grad_rf.cpu().numpy(), grad_c.cpu().numpy() / 1000.0
    dd.close()
    r32, c32, _ = O.das_adjoint(g, rf, w.fs_hz, TINY, c_mm, N.WINDOW_HAMMING, gi.astype(np.float64), precision=32)
    # the same shares in another order, at most 64 per sample: 64 x 2^-24 normwise
    assert np.linalg.norm(got_rf - r32) <= 4e-6 * np.linalg.norm(r32)
    parts = np.linalg.norm(r32) * np.linalg.norm(rf) * 150 / c_mm[0]
    assert abs(got_c[0] - c32[0]) <= 4e-6 * max(abs(c32[0]), parts)
