"""The context's dt-space tables are replaced only after every launch that
reads them, whatever stream it is on: calls with alternating speeds of sound on
two streams, and a captured call whose graph is replayed between eager ones."""
from dataclasses import replace

import pytest

from supra_amd import _native as N
from supra_amd import workloads as W
from supra_amd.beamformer import RxBeamformer, USRawData

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")

SPEEDS = (1480e3, 1540e3, 1600e3)


def setup():
    w = W.linear_2d(num_scatterers=20)
    w = replace(w, bf=replace(w.bf, num_scanlines=(64, 1)))
    g = w.geometry()
    raw = USRawData(torch.from_numpy(w.rf_host()).cuda(), w.fs_hz, g)
    return g, raw


def beamform(bf, raw, c, out=None, stream=None, window=N.WINDOW_HAMMING):
    return bf.perform_rx_beamforming(N.BF_DELAY_AND_SUM, raw, 1.0, c, window, 0.0, False, 0, out=out, stream=stream).data


def test_alternating_speeds_on_two_streams(device):
    g, raw = setup()
    want = {}
    for c in SPEEDS:
        bf = RxBeamformer(g)
        want[c] = beamform(bf, raw, c).clone()
        torch.cuda.synchronize()
        bf.close()
    bf = RxBeamformer(g)
    streams = [torch.cuda.Stream(), torch.cuda.Stream()]
    torch.cuda.synchronize()
    outs = []
    for i in range(24):
        c = SPEEDS[(i // 3) % 3]      # three launches, on both streams, before each change
        out = torch.empty_like(want[c])
        torch.cuda.synchronize()
        for _ in range(4):
            beamform(bf, raw, c, out=out, stream=streams[i % 2])
        outs.append((c, out))
    torch.cuda.synchronize()
    for i, (c, out) in enumerate(outs):
        assert torch.equal(out, want[c]), f"call {i}"
    bf.close()


def test_captured_call_replays(device):
    g, raw = setup()
    bf = RxBeamformer(g)
    c = SPEEDS[1]
    want = beamform(bf, raw, c).clone()
    rect = beamform(bf, raw, c, window=N.WINDOW_RECTANGULAR).clone()
    torch.cuda.synchronize()
    out = torch.zeros_like(want)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        beamform(bf, raw, c, out=out)
    for _ in range(3):
        out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want)
        assert torch.equal(beamform(bf, raw, c, window=N.WINDOW_RECTANGULAR), rect)
    bf.close()
