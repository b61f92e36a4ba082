"""Delays that are not finite numbers: a NaN in a scanline's geometry.  A NaN
delay converts to sample 0 with a NaN fraction, so with float RF (and with any
RF in 3D) every pixel of that scanline that has an element in its aperture
saturates; int16 RF in 2D leaves the element out.  An infinite delay is past
the last sample and adds nothing.  The other scanlines keep their bits."""
from dataclasses import replace

import numpy as np
import pytest

from oracle import oracle as O
from supra_amd import _native as N
from supra_amd import workloads as W
from supra_amd.beamformer import (RawDelay, RxBeamformer, USRawData, mv_das_perform_rx_beamforming,
                                  mv_perform_rx_beamforming)

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")

LINE = 4
LOWEST = -np.finfo(np.float32).max


def linear(elements=37, lines=9, depths=150):
    w = W.linear_2d(num_scatterers=1)
    return replace(w, bf=replace(w.bf, element_layout=(elements, 1), num_scanlines=(lines, 1), max_aperture=(elements, 1),
                                 tx_max_aperture=(elements, 1), num_depths=depths), num_channels=elements, num_samples=2400)


def broken(g, value, field="initial_delay"):
    scan = g.scanlines.copy()
    if field == "initial_delay":
        scan["tx"]["initial_delay"][LINE] = value
    else:
        scan["direction"][LINE, 1] = value      # depth component: coordinates whose squares overflow
    return replace(g, scanlines=scan)


def image(g, rf, kind, fs):
    eng = RxBeamformer(g)
    img = eng.perform_rx_beamforming(kind, USRawData(rf, fs, g), 1.0, 1540e3, N.WINDOW_RECTANGULAR, 0.0, False, 0)
    torch.cuda.synchronize()
    out = img.data.cpu().numpy()
    eng.close()
    return out


def check(clean, nan, inf, far_away, saturates):
    """`clean` of constant RF is 0 exactly where a pixel has no element."""
    member = clean[..., LINE] != 0
    assert member.any()
    want = np.where(member, np.float32(LOWEST if saturates else 0.0), np.float32(0.0))
    assert np.array_equal(nan[..., LINE], want)
    assert (inf[..., LINE] == 0).all()
    assert (far_away[..., 1:, LINE] == 0).all()
    others = np.arange(clean.shape[-1]) != LINE
    for img in (nan, inf, far_away):
        assert np.array_equal(img[..., others], clean[..., others])


@pytest.mark.parametrize("mapped", [False, True])
@pytest.mark.parametrize("dtype,frames", [(torch.int16, 1), (torch.float32, 1), (torch.float32, 3)])
def test_das_2d(device, dtype, frames, mapped):
    w = linear()
    g = w.geometry()
    if mapped:
        g = replace(g, element_to_channel=np.arange(37, dtype=np.int32)[::-1].copy())
    rf = torch.full((frames, *w.rf_shape), 7, dtype=dtype, device="cuda")
    args = (rf, N.BF_DELAY_AND_SUM, w.fs_hz)
    check(image(g, *args), image(broken(g, np.nan), *args), image(broken(g, np.inf), *args),
          image(broken(g, 1e30, "direction"), *args), dtype == torch.float32)


def test_batch(device):
    from supra_amd.batch import DAS, Batch
    w = linear()
    g = broken(w.geometry(), np.nan)
    rf = torch.full(w.rf_shape, 7.0, device="cuda")
    out = torch.zeros((g.num_depths, g.num_rx), device="cuda")
    b = Batch([dict(engine=RxBeamformer(g), rf=rf, out=out, fs_hz=w.fs_hz, mode=DAS,
                    window_type=N.WINDOW_RECTANGULAR)], autotune=False)
    b.launch()
    torch.cuda.synchronize()
    assert np.array_equal(out.cpu().numpy(), image(g, rf, N.BF_DELAY_AND_SUM, w.fs_hz))
    b.close()


@pytest.mark.parametrize("lx,ly", [(7, 5), (6, 40)])      # rows in registers; the general kernel
@pytest.mark.parametrize("dtype", [torch.int16, torch.float32])
def test_das_3d(device, dtype, lx, ly):
    w = W.matrix_3d_small(n_el=max(lx, ly), n_lines=4, n_depths=150, n_samples=1300)
    w = replace(w, bf=replace(w.bf, element_layout=(lx, ly), max_aperture=(lx, ly), tx_max_aperture=(lx, ly)),
                num_channels=lx * ly)
    g = w.geometry()
    args = (torch.full(w.rf_shape, 7, dtype=dtype, device="cuda"), N.BF_DELAY_AND_SUM, w.fs_hz)
    check(image(g, *args), image(broken(g, np.nan), *args), image(broken(g, np.inf), *args),
          image(broken(g, 1e30, "direction"), *args), True)


@pytest.mark.parametrize("kind", [N.BF_DELAY_AND_STD_DEV, N.BF_COHERENCE_FACTOR])
def test_variants(device, kind):
    w = linear()
    g = w.geometry()
    rf = torch.arange(1, 1 + np.prod(w.rf_shape), device="cuda").remainder(97).to(torch.float32).reshape(w.rf_shape)
    args = (rf, kind, w.fs_hz)
    clean, nan = image(g, *args), image(broken(g, np.nan), *args)
    member = image(g, torch.full(w.rf_shape, 7.0, device="cuda"), N.BF_DELAY_AND_SUM, w.fs_hz)[:, LINE] != 0
    assert np.array_equal(nan[:, LINE], np.where(member, np.float32(LOWEST), np.float32(0)))
    others = np.arange(clean.shape[1]) != LINE
    assert np.array_equal(nan[:, others], clean[:, others])


@pytest.mark.parametrize("dims", [2, 3])
@pytest.mark.parametrize("dtype", [np.int16, np.float32])
def test_nan_positions(device, dtype, dims):
    """An element whose position is NaN is in no aperture, and no element is in
    that of a scanline whose position is NaN: as the FP32 oracle."""
    w = linear() if dims == 2 else W.matrix_3d_small(n_el=6, n_lines=4, n_depths=150, n_samples=1300)
    g = w.geometry()
    ex, scan = g.element_x.copy(), g.scanlines.copy()
    ex[8] = np.nan
    scan["position"][1, 0] = np.nan
    g = replace(g, element_x=ex, scanlines=scan)
    rf = np.random.default_rng(0).integers(-2000, 2000, w.rf_shape).astype(dtype)
    for kind in (N.BF_DELAY_AND_SUM, N.BF_COHERENCE_FACTOR):
        ref = O.das(g, rf, w.fs_hz, 1.0, 1540e3, N.WINDOW_RECTANGULAR, sample_beamformer=kind)
        assert np.array_equal(image(g, torch.from_numpy(rf).cuda(), kind, w.fs_hz), ref)


@pytest.mark.parametrize("dtype", [torch.int16, torch.float32])
def test_pre_delay(device, dtype):
    """The pre-delayed element is -FLT_MAX (float RF), and the fused
    minimum variance sees the same data as the two calls."""
    w = linear(elements=24, lines=6, depths=90)
    g, bad = w.geometry(), broken(w.geometry(), np.nan)
    rf = torch.full(w.rf_shape, 7, dtype=dtype, device="cuda")
    out = []
    for geom in (g, bad):
        d = RawDelay(geom)
        out.append(d.perform_delay(USRawData(rf, w.fs_hz, geom), 1.0, 1540e3, N.WINDOW_RECTANGULAR, 0.0).data)
        d.close()
    clean, nan = (o.cpu().numpy() for o in out)
    want = np.where((clean[LINE] != 0) & (dtype == torch.float32), np.float32(LOWEST), np.float32(0))
    assert np.array_equal(nan[LINE], want)
    assert np.array_equal(np.delete(nan, LINE, 0), np.delete(clean, LINE, 0))
    eng = RxBeamformer(bad)
    fused = mv_das_perform_rx_beamforming(eng, USRawData(rf, w.fs_hz, bad), 1.0, 1540e3, N.WINDOW_RECTANGULAR, 0.0, 8, 2,
                                          1.5, False, 0.1).data
    steps = mv_perform_rx_beamforming(USRawData(out[1], 1.0, None, 1, (1, 1)), 8, 2, 1.5, False, 0.1).data
    assert torch.equal(fused, steps)
    eng.close()


def test_adjoint(device):
    """A gradient that reaches such a pixel is NaN at samples 0 and 1 of the
    elements of that scanline's transmit."""
    from supra_amd.differentiable import DifferentiableDAS
    w = linear(elements=24, lines=6, depths=90)
    g = w.geometry()
    rf = torch.randn((1, *w.rf_shape), generator=torch.Generator().manual_seed(0)).cuda()
    c = torch.tensor([1540.0], dtype=torch.float64, device="cuda")
    gi = torch.ones((1, 90, 6), device="cuda")
    a, b = (DifferentiableDAS(geom, w.fs_hz, 1.0, N.WINDOW_RECTANGULAR) for geom in (g, broken(g, np.nan)))
    _, norm = a.forward_raw(rf, c)
    clean, _ = a.adjoint_raw(rf, c, norm, gi)
    got, _ = b.adjoint_raw(rf, c, norm, gi)
    clean, got = clean.cpu().numpy()[0], got.cpu().numpy()[0]
    tx = int(g.scanlines["tx"]["tx_idx"][LINE, np.argmax(g.scanlines["tx_weights"][LINE])])
    used = (clean[tx] != 0).any(axis=1)
    assert used.any() and np.isnan(got[tx][used, :2]).all() and (got[tx][used, 2:] == 0).all()
    assert np.array_equal(np.delete(got, tx, 0), np.delete(clean, tx, 0))
    a.close()
    b.close()
