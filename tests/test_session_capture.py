"""Batched sessions under stream capture (``-m gpu``).

At shapes whose batches only share launches, a graph of a batch runs its sessions one by one, each in
the workspace an earlier eager batch sized for it. So nothing another batch of the same prefix does
later (growing the prefix's own workspace, running on another stream) reaches the graph: its replays
are the sessions' own calls bit for bit (the same launches)."""

import ctypes as C

import numpy as np
import pytest

import kivi
from helpers import DeviceArrays
from kivi import KiviCache, KiviConfig

pytestmark = pytest.mark.gpu

SCALE = np.float32(0.1)


class Rig:
    def __init__(self, amd, bits=4, group=32, dim=96, heads=2, gq=2, n=900, residual=None):
        self.amd, self.heads, self.dim, self.qh = amd, heads, dim, heads * gq
        self.per = self.qh * dim
        self.rng = np.random.default_rng(7700 + dim + group)
        self.hip = C.CDLL("libamdhip64.so.7")
        self.mem = DeviceArrays()
        self.cache = KiviCache(amd, KiviConfig(bits, group, residual or 2 * group), 1, heads, dim)
        self.cache.append(*self.rows(n), n)
        self.prefix = self.cache.share_prefix()

    def rows(self, n):
        return [self.rng.standard_normal((self.heads, n, self.dim)).astype(np.float32) for _ in range(2)]

    def sessions(self, lengths):
        out = []
        for n in lengths:
            s = self.prefix.session()
            if n:
                s.append(*self.rows(n), n)
            out.append(s)
        return out

    def batch(self, sessions):
        """Queries of a batch, its device buffers and each session's own result."""
        q = self.rng.standard_normal(len(sessions) * self.per).astype(np.float32)
        want = np.concatenate([s.attention(q[i * self.per:(i + 1) * self.per], self.qh, SCALE)
                               for i, s in enumerate(sessions)])
        return Batch(self, sessions, self.mem.upload(q), self.mem.empty(q.size), want)

    def stream(self):
        s = C.c_void_p()
        assert self.hip.hipStreamCreate(C.byref(s)) == 0
        return s

    def wait(self, stream):
        assert self.hip.hipStreamSynchronize(stream) == 0


class Batch:
    def __init__(self, rig, sessions, dq, out, want):
        self.rig, self.sessions, self.dq, self.out, self.want = rig, sessions, dq, out, want

    def call(self, stream):
        n = len(self.sessions) * self.rig.per
        kivi.sessions_attention_device(self.rig.amd, self.sessions, self.dq, n, self.rig.qh, SCALE, self.out, n,
                                       stream.value)

    def eager(self, stream):
        self.call(stream)
        self.rig.wait(stream)
        assert np.abs(self.result() - self.want).max() < 2e-4  # other splits than the sessions' own

    def capture(self, stream):
        hip = self.rig.hip
        graph, exe = C.c_void_p(), C.c_void_p()
        assert hip.hipStreamBeginCapture(stream, 0) == 0  # global mode: an allocation is refused
        try:
            self.call(stream)
        finally:
            rc = hip.hipStreamEndCapture(stream, C.byref(graph))
        assert rc == 0
        assert hip.hipGraphInstantiate(C.byref(exe), graph, None, None, C.c_size_t(0)) == 0
        assert hip.hipGraphDestroy(graph) == 0
        return exe

    def clear(self):
        zero = np.zeros(self.want.size, np.float32)
        assert self.rig.hip.hipMemcpy(C.c_void_p(self.out), zero.ctypes.data_as(C.c_void_p), C.c_size_t(zero.nbytes), 1) == 0

    def result(self):
        return self.rig.mem.download(self.out, self.want.size)


SHAPES = [(4, 32, 96, 2), (2, 64, 128, 4), (4, 8, 64, 1), (8, 32, 192, 2)]  # lanes, chunks, rows, chunks and rows


@pytest.mark.parametrize("bits,group,dim,gq", SHAPES)
def test_graph_outlives_a_larger_batch(amd, bits, group, dim, gq):
    """Captured after its own eager batch; then a larger batch of other sessions and another cache."""
    r = Rig(amd, bits, group, dim, 2, gq)
    small = r.batch(r.sessions([0, 17, 70]))
    large = r.batch(r.sessions([300 + 11 * i for i in range(14)]))
    stream = r.stream()
    small.eager(stream)
    exe = small.capture(stream)
    large.eager(stream)
    others = []
    for n in (600, 900, 1500):
        c = KiviCache(amd, KiviConfig(bits, group, 2 * group), 1, 2, dim)
        c.append(*r.rows(n), n)
        others.append((c, [np.asarray(x).view(np.uint32).copy() for x in c.export_streams()]))
    for _ in range(3):
        small.clear()
        assert r.hip.hipGraphLaunch(exe, stream) == 0
        r.wait(stream)
        assert np.array_equal(small.result().view(np.uint32), small.want.view(np.uint32))
        large.eager(stream)
    for c, streams in others:
        assert all(np.array_equal(np.asarray(x).view(np.uint32), y) for x, y in zip(c.export_streams(), streams))
    assert r.hip.hipGraphExecDestroy(exe) == 0 and r.hip.hipStreamDestroy(stream) == 0
    r.mem.free()


@pytest.mark.parametrize("bits,group,dim,gq", SHAPES)
def test_graphs_of_disjoint_sessions_replay_side_by_side(amd, bits, group, dim, gq):
    """Two batches, each warmed and captured on its own stream (the second's warm-up lies between the
    first's and its capture, and the sessions' own calls ran on the default stream before)."""
    r = Rig(amd, bits, group, dim, 2, gq)
    batches = [r.batch(r.sessions([40 * i + b for i in range(5)])) for b in range(2)]
    streams = [r.stream() for _ in batches]
    for b, s in zip(batches, streams):
        b.eager(s)
    graphs = [b.capture(s) for b, s in zip(batches, streams)]
    for _ in range(5):
        for b in batches:
            b.clear()
        for _ in range(4):
            for exe, s in zip(graphs, streams):
                assert r.hip.hipGraphLaunch(exe, s) == 0
        for s in streams:
            r.wait(s)
        for b in batches:
            assert np.array_equal(b.result().view(np.uint32), b.want.view(np.uint32))
    for exe, s in zip(graphs, streams):
        assert r.hip.hipGraphExecDestroy(exe) == 0 and r.hip.hipStreamDestroy(s) == 0
    r.mem.free()


@pytest.mark.parametrize("gq,most", [(1, 9), (2, 9), (4, 5), (8, 3)])
def test_fewer_sessions_than_warmed(amd, gq, most):
    """head_dim 128 and group 32, where a graph keeps the prefix's workspace: an eager batch sizes it for
    every smaller batch of the prefix too (fewer rows take more splits of the chunks)."""
    r = Rig(amd, 2, 32, 128, 8, gq, 10007)
    sessions = r.sessions([0, 17, 70, 140, 30, 9, 0, 64, 5][:most])
    stream = r.stream()
    r.batch(sessions).eager(stream)
    for count in range(most, 0, -1):
        b = r.batch(sessions[:count])
        exe = b.capture(stream)
        for _ in range(3):
            b.clear()
            assert r.hip.hipGraphLaunch(exe, stream) == 0
            r.wait(stream)
            assert np.abs(b.result() - b.want).max() < 2e-4
        assert r.hip.hipGraphExecDestroy(exe) == 0
    assert r.hip.hipStreamDestroy(stream) == 0
    r.mem.free()


def test_fewer_sessions_than_warmed_behind_a_long_window(amd):
    """A residual of 2048 tokens: 40 sessions run as a GEMM, few of them in groups of 16 rows, and the
    captured ones have shorter suffixes than the batch that sized the workspace."""
    r = Rig(amd, 2, 32, 128, 8, 1, 10007, 2048)
    sessions = r.sessions(sorted((29 * i) % 150 for i in range(40)))
    stream = r.stream()
    r.batch(sessions).eager(stream)
    for count in [40, 33, 31, 24, 20, 17, 16, 15, 12, 9, 6, 4, 3, 2, 1]:
        b = r.batch(sessions[:count])
        exe = b.capture(stream)
        for _ in range(3):
            b.clear()
            assert r.hip.hipGraphLaunch(exe, stream) == 0
            r.wait(stream)
            assert np.abs(b.result() - b.want).max() < 2e-4
        assert r.hip.hipGraphExecDestroy(exe) == 0
    assert r.hip.hipStreamDestroy(stream) == 0
    r.mem.free()
