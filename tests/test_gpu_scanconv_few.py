"""2D scan conversion of few frames, where the form changes from one pixel per
thread to staged tiles: every frame holds the bits that it has in a
launch of many frames."""
import pytest

from supra_amd.geometry import BeamformerConfig, RxGeometry
from supra_amd.scanconv import ScanConverter

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


@pytest.mark.parametrize("in_dtype,out_dtype", [("uint8", "uint8"), ("float32", "int16"), ("int16", "float32")])
@pytest.mark.parametrize("sector,lines,depths,res", [(0.0, 2, 2, 0.31), (0.0, 61, 301, 0.17), (60.0, 97, 403, 0.13)])
def test_few_frames(device, sector, lines, depths, res, in_dtype, out_dtype):
    kw = {} if sector == 0.0 else dict(scan_type="phased", sector_angle_deg=(sector, 0.0))
    elements = 128 if sector else lines
    cfg = BeamformerConfig(element_layout=(elements, 1), num_scanlines=(lines, 1), max_aperture=(elements, 1),
                           tx_max_aperture=(elements, 1), depth=30.0, num_depths=depths, **kw)
    sc = ScanConverter()
    sc.update_internals(RxGeometry.from_config(cfg), depths, res)
    g = torch.Generator(device="cuda").manual_seed(lines)
    images = (torch.rand((21, depths, lines), generator=g, device="cuda") * 250.0).to(getattr(torch, in_dtype))
    out_dtype = getattr(torch, out_dtype)
    many = sc.convert(images, out_dtype)
    for count in (1, 3, 4, 5, 20):
        for first in range(0, 22 - count, count):
            few = sc.convert(images[first:first + count].contiguous(), out_dtype)
            assert torch.equal(few, many[first:first + count]), (count, first)
