"""The minimum variance of well-loaded systems does not depend on the plan: the
depth tile that a launch or a batch plans for its share of the LDS changes no
bit.  The test program built next to the library plans every configuration for
an eighth to all of the LDS; batches of 128-element acquisitions (windows of
many sub-array vectors) equal the single calls, with and without tuning."""
import subprocess
from pathlib import Path

import numpy as np
import pytest

from supra_amd import _native as N
from supra_amd import workloads as W
from supra_amd.beamformer import RxBeamformer, USRawData, mv_das_perform_rx_beamforming

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")

PROG = Path(__file__).resolve().parent.parent / "supra_amd" / "mv_plans_test"


def test_every_plan_gives_the_same_bits(device):
    if not PROG.exists():
        pytest.fail(f"{PROG} is missing: build the library (python -m supra_amd.build)")
    res = subprocess.run([str(PROG)], capture_output=True, text=True, timeout=100)
    print(res.stdout)
    assert res.returncode == 0 and res.stdout.count(", 0 failures") == 11, res.stdout + res.stderr


@pytest.mark.parametrize("autotune", [False, True])
def test_batch_of_wide_apertures(device, autotune):
    from supra_amd.batch import MV, Batch
    items, refs = [], []
    for i, (n_d, L, T, dtype) in enumerate([(290, 64, 5, np.int16), (203, 64, 2, np.int16), (311, 32, 5, np.float32),
                                            (150, 16, 4, np.float32)]):
        w = W.linear_acquisition(140, n_d, 128, 40e6, 60, scatter_seed=5 + i, noise_seed=8 + i)
        g = w.geometry()
        rf = torch.from_numpy(w.rf_host(dtype=dtype)).cuda()
        eng = RxBeamformer(g)
        out = torch.full((g.num_depths, g.num_rx), -7.0, device="cuda")
        items.append(dict(engine=eng, rf=rf, out=out, fs_hz=40e6, mode=MV, f_number=0.3, sub_array_size=L,
                          temporal_smoothing=T, loading_factor=0.01))
        refs.append(mv_das_perform_rx_beamforming(eng, USRawData(rf, 40e6, g), 0.3, 1540e3, N.WINDOW_HANN, 0.0, L, T,
                                                  1.5, False, 0.01).data)
    b = Batch(items, autotune=autotune)
    print(b.config())
    b.launch()
    torch.cuda.synchronize()
    for it, ref in zip(items, refs):
        assert torch.equal(it["out"], ref)
    b.close()
