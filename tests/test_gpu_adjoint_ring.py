"""The adjoint kernel's chunk and ring rules against the FP32 oracle's reverse
mode (same arithmetic, another summation order): depth counts around the
64-depth chunk, odd apertures (a wave with one element only), so many depths
that three share a sample, so few that a chunk is wider than the ring, delays
below the first and past the last sample, lines with several writers, and
pixels without gradient."""
from dataclasses import replace

import numpy as np
import pytest

from oracle import oracle as O
from supra_amd import workloads as W

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")

# A sample of dL/drf sums at most ~2 shares per lane and element writer (below
# 64 here) and dL/dc's slots 40 chunks per lane before they go on in double:
# 64 roundings of 2^-24, 4e-6, normwise.
TOL = 1e-5


@pytest.mark.parametrize("elements,lines,depths,samples,offset,sparse,shared", [
    (31, 5, 63, 2080, 0, False, False),
    (32, 5, 64, 2080, -40, False, False),
    (33, 4, 65, 1111, 0, True, False),
    (64, 3, 2500, 701, 6, False, False),      # three and more depths per sample
    (17, 3, 40, 4097, -900, False, False),    # tens of samples per depth
    (48, 6, 1000, 1500, 250, True, True),     # two elements per channel
    (3, 2, 130, 64, 0, False, False),
])
def test_chunks_and_rings(device, elements, lines, depths, samples, offset, sparse, shared):
    from supra_amd.differentiable import DifferentiableDAS
    w = W.linear_2d(num_scatterers=1)
    w = replace(w, bf=replace(w.bf, element_layout=(elements, 1), num_scanlines=(lines, 1), max_aperture=(elements, 1),
                              tx_max_aperture=(elements, 1), num_depths=depths), num_channels=elements)
    g = w.geometry()
    channels = (elements + 1) // 2 if shared else elements
    rng = np.random.default_rng(elements * 7 + depths)
    if sparse or shared:
        emap = (np.arange(elements) % channels).astype(np.int32)
        if sparse:
            emap[rng.choice(elements, elements // 5, replace=False)] = -1
        g.element_to_channel = emap
    c_mm = np.array([1480.0e3, 1560.0e3])
    rf = rng.normal(size=(2, lines, channels, samples)).astype(np.float32)
    gi = rng.normal(size=(2, depths, lines)).astype(np.float32)
    gi[:, ::7] = 0.0
    a = w.das_kwargs()
    dd = DifferentiableDAS(g, w.fs_hz, a["f_number"], a["window_type"], a["window_parameter"], False, offset)
    x = torch.from_numpy(rf).cuda()
    c = torch.tensor(c_mm / 1000.0, dtype=torch.float64, device="cuda")
    _, norm = dd.forward_raw(x, c)
    grad_rf, grad_c = dd.adjoint_raw(x, c, norm, torch.from_numpy(gi).cuda())
    torch.cuda.synchronize()
    # either gradient alone is the same (one writer per line: the same sums)
    alone_rf, none = dd.adjoint_raw(x, c, norm, torch.from_numpy(gi).cuda(), want_c=False)
    assert none is None and (shared or torch.equal(alone_rf, grad_rf))
    none, alone_c = dd.adjoint_raw(x, c, norm, torch.from_numpy(gi).cuda(), want_rf=False)
    assert none is None and torch.equal(alone_c, grad_c)
    got_rf, got_c = grad_rf.cpu().numpy(), grad_c.cpu().numpy() / 1000.0
    dd.close()
    r32, c32, _ = O.das_adjoint(g, rf, w.fs_hz, a["f_number"], c_mm, a["window_type"], gi.astype(np.float64),
                                a["window_parameter"], False, offset, precision=32)
    scale = np.linalg.norm(r32)
    assert np.linalg.norm(got_rf - r32) <= TOL * scale
    assert np.all(got_rf[r32 == 0] == 0)
    # the terms of dL/dc cancel: relative to the norm of its gradient's parts
    parts = np.array([np.linalg.norm(r32[f]) * np.linalg.norm(rf[f]) * depths / c_mm[f] for f in range(2)])
    assert np.all(np.abs(got_c - c32) <= TOL * np.maximum(np.abs(c32), parts))
