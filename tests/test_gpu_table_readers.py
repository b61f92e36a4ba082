"""Who a call with another speed of sound waits for before it replaces the
context's tables.  Every test keeps a stream busy with a bounded sleep in front
of the launch that reads the old tables, so that the launch has not begun when
the next call comes: without the wait it would find the new tables."""
from dataclasses import replace

import pytest

from supra_amd import _native as N
from supra_amd import workloads as W
from supra_amd.beamformer import RxBeamformer, USRawData

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")

OLD, NEW = 1480e3, 1600e3
BUSY_MS = 60.0


class Calls:
    def __init__(self):
        w = W.linear_2d(num_scatterers=20)
        w = replace(w, bf=replace(w.bf, num_scanlines=(64, 1)))
        g = w.geometry()
        self.raw = USRawData(torch.from_numpy(w.rf_host()).cuda(), w.fs_hz, g)
        self.want = {}
        for c in (OLD, NEW):
            self.bf = RxBeamformer(g)
            self.want[c] = self(c, self.out(g), None).clone()
            torch.cuda.synchronize()
            self.bf.close()
        self.bf = RxBeamformer(g)
        self.outs = [self.out(g) for _ in range(20)]
        # cycles of a sleep of BUSY_MS
        a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        torch.cuda._sleep(1000)
        a.record()
        torch.cuda._sleep(1_000_000)
        b.record()
        torch.cuda.synchronize()
        self.cycles = int(1_000_000 * BUSY_MS / max(a.elapsed_time(b), 1e-3))

    @staticmethod
    def out(g):
        return torch.zeros((g.num_depths, g.num_rx), device="cuda")

    def __call__(self, c, out, stream):
        return self.bf.perform_rx_beamforming(N.BF_DELAY_AND_SUM, self.raw, 1.0, c, N.WINDOW_HAMMING, 0.0, False, 0, out=out,
                                              stream=stream).data

    def busy(self, stream):
        with torch.cuda.stream(stream):
            torch.cuda._sleep(self.cycles)

    def check(self, c, out):
        assert torch.equal(out, self.want[c])


@pytest.fixture()
def calls(device):
    k = Calls()
    yield k
    torch.cuda.synchronize()
    k.bf.close()


def test_readers_on_another_stream(calls):
    a, b = torch.cuda.Stream(), torch.cuda.Stream()
    calls(OLD, calls.outs[0], a)
    torch.cuda.synchronize()
    calls.busy(a)
    calls(OLD, calls.outs[1], a)
    calls(NEW, calls.outs[2], b)
    torch.cuda.synchronize()
    calls.check(OLD, calls.outs[1])
    calls.check(NEW, calls.outs[2])


def test_readers_on_the_same_stream(calls):
    a = torch.cuda.Stream()
    calls(OLD, calls.outs[0], a)
    calls.busy(a)
    calls(OLD, calls.outs[1], a)
    calls(NEW, calls.outs[2], a)
    torch.cuda.synchronize()
    calls.check(OLD, calls.outs[1])
    calls.check(NEW, calls.outs[2])


def test_readers_on_more_streams_than_are_noted(calls):
    streams = [torch.cuda.Stream() for _ in range(18)]
    assert len({s.cuda_stream for s in streams}) == 18
    for s, out in zip(streams, calls.outs):
        calls(OLD, out, s)
    torch.cuda.synchronize()
    for s in streams[:-1]:
        calls(OLD, calls.outs[0], s)
    torch.cuda.synchronize()
    calls.outs[17].zero_()
    torch.cuda.synchronize()
    calls.busy(streams[17])
    calls(OLD, calls.outs[17], streams[17])
    calls(NEW, calls.outs[18], streams[0])
    torch.cuda.synchronize()
    calls.check(OLD, calls.outs[17])
    calls.check(NEW, calls.outs[18])


def test_a_replay_in_flight(calls):
    """A captured call reads the tables when it is replayed, on a stream that
    no call was made on."""
    a, b = torch.cuda.Stream(), torch.cuda.Stream()
    calls(OLD, calls.outs[0], a)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        calls(OLD, calls.outs[1], None)
    for _ in range(2):
        calls(OLD, calls.outs[0], a)
        torch.cuda.synchronize()
        calls.outs[1].zero_()
        torch.cuda.synchronize()
        calls.busy(b)
        with torch.cuda.stream(b):
            graph.replay()
        calls(NEW, calls.outs[2], a)
        torch.cuda.synchronize()
        calls.check(OLD, calls.outs[1])
        calls.check(NEW, calls.outs[2])


def test_other_work_is_not_waited_for(calls):
    a, b, other = (torch.cuda.Stream() for _ in range(3))
    done = torch.cuda.Event()
    calls(OLD, calls.outs[0], a)
    calls.busy(other)
    done.record(other)
    calls(NEW, calls.outs[1], b)
    assert not done.query(), "the call waited for a stream without work of this context"
    torch.cuda.synchronize()
    calls.check(OLD, calls.outs[0])
    calls.check(NEW, calls.outs[1])
