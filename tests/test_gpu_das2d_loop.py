"""The 2D loop's range rules against the FP32 oracle, bit for bit: receive
data of one and two samples and of a ragged length, offsets that push delays
below the first and past the last sample, non-finite samples, unconnected
channels, apertures wider than one staged chunk of elements whose near field
starts and ends inside it, delay-and-sum and coherence factor."""
from dataclasses import replace

import numpy as np
import pytest

from oracle import oracle as O
from supra_amd import _native as N
from supra_amd import workloads as W
from supra_amd.beamformer import RxBeamformer, USRawData

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


@pytest.mark.parametrize("kind", [N.BF_DELAY_AND_SUM, N.BF_COHERENCE_FACTOR])
@pytest.mark.parametrize("elements,lines,depths,samples,offset,dtype,sparse", [
    (128, 9, 200, 1, 0, np.int16, False),
    (128, 9, 200, 2, -3, np.float32, False),
    (37, 5, 130, 701, -400, np.int16, True),
    (192, 7, 333, 1501, 0, np.float32, False),
    (192, 7, 333, 1501, 300, np.int16, True),
    (300, 3, 65, 2049, -100000, np.float32, True),
])
def test_2d_ranges(device, kind, elements, lines, depths, samples, offset, dtype, sparse):
    w = W.linear_2d(num_scatterers=1)
    w = replace(w, bf=replace(w.bf, element_layout=(elements, 1), num_scanlines=(lines, 1), max_aperture=(elements, 1),
                              tx_max_aperture=(elements, 1), num_depths=depths), num_channels=elements)
    g = w.geometry()
    rng = np.random.default_rng(elements + samples)
    rf = rng.integers(-2000, 2000, (lines, elements, samples)).astype(dtype)
    if dtype == np.float32:
        rf += rng.random(rf.shape, dtype=np.float32)
        rf[0, ::3, samples - 1] = np.inf
        rf[lines - 1, ::5, samples // 2] = np.nan
    if sparse:
        emap = np.arange(elements, dtype=np.int32)
        emap[rng.choice(elements, elements // 6, replace=False)] = -1
        g.element_to_channel = emap
    kw = dict(w.das_kwargs(), additional_offset=offset)
    bf = RxBeamformer(g)
    img = bf.perform_rx_beamforming(kind, USRawData(torch.from_numpy(rf).cuda(), w.fs_hz, g), kw["f_number"],
                                    kw["speed_of_sound_mm_per_s"], kw["window_type"], 0.0, False, offset)
    torch.cuda.synchronize()
    got = img.data.cpu().numpy()
    bf.close()
    ref = O.das(g, rf, w.fs_hz, sample_beamformer=kind, **kw)
    ok = (got == ref) | (np.isnan(got) & np.isnan(ref))
    assert ok.all(), f"{(~ok).sum()} of {ok.size} pixels differ"
