"""Both sides of the rule between the two 3D kernels: volumes that fill the card
together (the general kernel) hold the bits that each has alone (the kernel for
separable grids), which are the FP32 oracle's."""
import numpy as np
import pytest

from oracle import oracle as O
from supra_amd import workloads as W
from supra_amd.beamformer import RxBeamformer, USRawData

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


@pytest.mark.parametrize("dtype", [np.int16, np.float32])
@pytest.mark.parametrize("offset", [0, 3])
def test_many_volumes_and_one(device, dtype, offset):
    w = W.matrix_3d_small(n_el=7, n_lines=8, n_depths=300, n_samples=900)   # 128 workgroups a volume
    g = w.geometry()
    kw = dict(w.das_kwargs(), additional_offset=offset)
    rf = np.random.default_rng(offset).integers(-20000, 20000, (10, *w.rf_shape)).astype(dtype)
    eng = RxBeamformer(g)

    def run(x):
        return eng.perform_rx_beamforming(0, USRawData(x, w.fs_hz, g), kw["f_number"], kw["speed_of_sound_mm_per_s"],
                                          kw["window_type"], kw["window_parameter"], False, offset).data

    x = torch.from_numpy(rf).cuda()
    together = run(x)
    alone = torch.stack([run(x[f]) for f in range(10)])
    torch.cuda.synchronize()
    assert torch.equal(together, alone)
    assert np.array_equal(alone[7].cpu().numpy(), O.das(g, rf[7], w.fs_hz, **kw))
    eng.close()
