"""The three forms of the 2D scan conversion (direct, runs of 1024 pixels, pixel
tiles) on either side of the frame counts and image sizes that choose between
them, bit for bit the oracle's arithmetic on the library's own tables: odd frame
counts, images around a tile and a run, dense sectors whose apex tiles do not fit
the window, outputs off the alignment that runs need, samples that are not
finite."""
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


def linear(lines, samples, depth, pitch=0.3):
    s = np.zeros(lines, SCANLINE_DTYPE)
    s["position"][:, 0] = np.arange(lines) * pitch
    s["direction"] = [0.0, 1.0, 0.0]
    return types.SimpleNamespace(scanlines=s, rx_layout=(lines, 1), depth=float(depth), num_depths=samples)


TYPES = {"u8": torch.uint8, "i16": torch.int16, "f32": torch.float32}


def check(g, res, frames, din, dout, shift):
    from supra_amd.scanconv import ScanConverter
    sc = ScanConverter()
    sc.update_internals(g, resolution=res)
    _, idx, w = sc.tables()
    rng = np.random.default_rng(frames)
    shape = (frames, g.num_depths, g.rx_layout[0])
    if din == "f32":
        img = (rng.normal(size=shape) * 300).astype(np.float32)
        img[rng.random(shape) < 0.002] = np.nan
        img[rng.random(shape) < 0.002] = np.inf
        img[:, g.num_depths // 2, :2] = -np.inf
    else:
        img = rng.integers(0, 256, shape).astype(np.uint8 if din == "u8" else np.int16)
    n = sc.num_pixels
    flat = torch.full((frames * n + 8,), 7, dtype=TYPES[dout], device="cuda")
    out = flat[shift:shift + frames * n].view(frames, sc.image_size[1], sc.image_size[0])
    sc.convert(torch.from_numpy(img).cuda(), TYPES[dout], out=out)
    torch.cuda.synchronize()
    assert (flat[:shift] == 7).all() and (flat[shift + frames * n:] == 7).all()
    got = out.cpu().numpy().reshape(frames, -1)
    tab = dict(size=sc.image_size, index=idx, weights=w, layout=g.rx_layout, is3d=False, num_samples=g.num_depths)
    with np.errstate(all="ignore"):
        want = SC.convert(tab, img, got.dtype.type)
    same = got == want
    assert same.all(), f"{(~same).sum()} pixels differ, first (frame, pixel) {np.argwhere(~same)[0]}"
    sc.close()


@pytest.mark.parametrize("din,dout", [("u8", "u8"), ("f32", "f32"), ("f32", "i16")])
@pytest.mark.parametrize("g,res,frames", [
    (linear(2, 30, 3.0), 0.1, 25), (linear(22, 61, 6.3), 0.1, 27), (linear(22, 62, 1.5), 0.1, 31),
    (linear(23, 200, 1.6), 0.1, 25), (linear(61, 301, 31.0), 0.17, 97),       # parallel: tiles
    (sector(40, 33, 101, 20.0), 0.21, 13), (sector(60, 301, 900, 12.0), 0.1, 13), (sector(30, 700, 400, 10.0), 0.17, 15),
    (sector(60, 301, 900, 60.0), 0.1, 9)])                                    # the last: more than 200,000 pixels
def test_tiles(device, g, res, frames, din, dout):
    check(g, res, frames, din, dout, 1)


@pytest.mark.parametrize("shift", [0, 1])       # 1: no packed stores, so no runs
@pytest.mark.parametrize("din,dout", [("u8", "u8"), ("i16", "f32"), ("f32", "f32"), ("f32", "u8")])
@pytest.mark.parametrize("g,res,frames", [
    (linear(7, 120, 1.5, 0.35), 0.0014, 5),             # 1501 x 1073 pixels or so, short runs
    (linear(250, 240, 10.0, 0.06), 0.0095, 11),         # 1573 x 1053, longer runs
    (linear(90, 500, 12.0, 0.1), 0.01, 22)])            # 891 x 1201
def test_runs(device, g, res, frames, din, dout, shift):
    from supra_amd.scanconv import ScanConverter
    # a resolution near `res` whose image goes out in fours
    for k in range(40):
        sc = ScanConverter()
        sc.update_internals(g, resolution=res * (1 + 0.001 * k))
        n = sc.num_pixels
        r = sc.resolution
        sc.close()
        if n % 4 == 0:
            break
    assert n % 4 == 0 and n >= 800000
    check(g, r, frames, din, dout, shift)
