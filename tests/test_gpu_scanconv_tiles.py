"""The tiled 2D scan conversion at the edges of its pixel tiles, frame pairs
and window, on the library's own tables: bit for bit the oracle's arithmetic."""
import types

import numpy as np
import pytest

from oracle import scanconv as SC
from supra_amd.geometry import SCANLINE_DTYPE

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


def sector(half_angle, lines, samples, depth):
    th = np.deg2rad(np.linspace(-half_angle, half_angle, lines))
    s = np.zeros(lines, SCANLINE_DTYPE)
    s["direction"] = np.stack([np.sin(th), np.cos(th), 0 * th], 1)
    return types.SimpleNamespace(scanlines=s, rx_layout=(lines, 1), depth=float(depth), num_depths=samples)


def linear(lines, samples, depth):
    s = np.zeros(lines, SCANLINE_DTYPE)
    s["position"][:, 0] = np.arange(lines) * 0.3
    s["direction"] = [0.0, 1.0, 0.0]
    return types.SimpleNamespace(scanlines=s, rx_layout=(lines, 1), depth=float(depth), num_depths=samples)


@pytest.mark.parametrize("case", [
    # (scan, resolution, frames): image widths around a tile, few and many
    # frames (odd counts leave half a pair), windows that hold a tile's box
    # everywhere, and dense sectors whose apex tiles do not fit
    (linear(2, 30, 3.0), 0.1, 1), (linear(22, 61, 6.3), 0.1, 2), (linear(22, 62, 1.5), 0.1, 3),
    (linear(23, 200, 1.6), 0.1, 7), (sector(40, 33, 101, 20.0), 0.21, 5), (sector(60, 301, 900, 12.0), 0.1, 2),
    (sector(30, 700, 400, 10.0), 0.17, 3)])
@pytest.mark.parametrize("dtype", ["u8", "f32"])
def test_tiles(device, case, dtype):
    from supra_amd.scanconv import ScanConverter
    g, res, frames = case
    sc = ScanConverter()
    sc.update_internals(g, resolution=res)
    mask, idx, w = sc.tables()
    rng = np.random.default_rng(frames)
    shape = (frames, g.num_depths, g.rx_layout[0])
    np_t, t_t = (np.uint8, torch.uint8) if dtype == "u8" else (np.float32, torch.float32)
    img = rng.integers(0, 256, shape).astype(np_t) if dtype == "u8" else rng.normal(size=shape).astype(np_t) * 1000
    # an output that starts off every vector alignment
    n = sc.num_pixels
    flat = torch.full((frames * n + 1,), 7, dtype=t_t, device="cuda")
    out = flat[1:].view(frames, sc.image_size[1], sc.image_size[0])
    sc.convert(torch.from_numpy(img).cuda(), t_t, out=out)
    torch.cuda.synchronize()
    got = out.cpu().numpy()
    assert flat[0].item() == 7
    tab = dict(size=sc.image_size, index=idx, weights=w, layout=g.rx_layout, is3d=False, num_samples=g.num_depths)
    want = SC.convert(tab, img, np_t)
    assert np.array_equal(got.reshape(frames, -1), want), f"{(got.reshape(frames, -1) != want).sum()} pixels differ"
    sc.close()
