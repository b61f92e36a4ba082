"""Minimum variance of at most 16 rows with long windows: tall depth tiles (32,
48 and 64 outputs, 8 to 16 per wave) of frames with enough of them, at the
edges of the rule, of tiles and of sub-blocks, against the FP64 oracle."""
import numpy as np
import pytest

from oracle import oracle as O
from test_gpu_mv_block import apertures, check, gpu_mv

pytestmark = pytest.mark.gpu
pytest.importorskip("torch")


@pytest.mark.parametrize("L,T,n_ch,n_rx,n_d,means", [
    (16, 4, 24, 48, 250, False), (1, 9, 20, 64, 170, True), (16, 6, 20, 384, 20, False),     # 32 outputs per tile
    (5, 10, 40, 64, 260, False), (13, 19, 33, 96, 157, True),                                # 48
    (16, 32, 170, 64, 330, False), (3, 12, 160, 64, 321, True), (13, 20, 33, 128, 157, True),  # 64
    (8, 32, 256, 64, 321, False)])                                                           # 64 do not fit
def test_tall_tiles(device, L, T, n_ch, n_rx, n_d, means):
    x = apertures(np.random.default_rng(L * 100 + T), n_rx, n_ch, n_d)
    check(gpu_mv(x, L, T, 1.5, means, 0.1), O.mv(x, L, T, 1.5, means, 0.1), L, 0.1)
