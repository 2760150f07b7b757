"""Device memory the library keeps between objects (``-m gpu``): a buffer given back and taken again
holds nothing of its previous owner, threads and streams share the pool, what it keeps is bounded,
and a call that would allocate is refused under stream capture as hipMalloc would be."""

import ctypes as C
import threading

import numpy as np
import pytest

import kivi
from kivi import KiviCache, KiviConfig, KiviError, quantize_per_channel
from helpers import DeviceArrays

pytestmark = pytest.mark.gpu


def rows(seed, units, n, dim, factor=1.0):
    rng = np.random.default_rng(seed)
    return [(rng.standard_normal((units, n, dim)) * factor).astype(np.float32) for _ in range(2)]


def streams_of(backend, seed, units, n, dim, bits=4):
    c = KiviCache(backend, KiviConfig(bits, 32, 32), 1, units, dim)
    k, v = rows(seed, units, n, dim)
    c.append(k, v, n)
    q = np.random.default_rng(seed + 1).standard_normal(units * 2 * dim).astype(np.float32)
    return [np.asarray(x).view(np.uint32).copy() for x in c.export_streams()], c.attention(q, 2 * units, 0.1)


@pytest.mark.parametrize("dim", [64, 96, 128])
def test_a_reused_buffer_shows_nothing_of_its_owner(amd, oracle, dim):
    units = 3
    for seed, n in enumerate((300, 37, 290, 70, 310)):
        loud = KiviCache(amd, KiviConfig(4, 32, 32), 1, units, dim)  # fills the buffers with NaN and inf
        k, v = rows(90 + seed, units, 320, dim, 1e30)
        k[:, :, 3] = np.nan
        v[:, :, 5] = np.inf
        loud.append(k, v, 320)
        del loud
        got, out = streams_of(amd, seed, units, n, dim)
        want, ref = streams_of(oracle, seed, units, n, dim)
        for x, y in zip(got, want):
            assert np.array_equal(x, y)
        assert np.abs(out - ref).max() < 1e-4


def test_threads_share_the_pool(amd):
    want = {s: streams_of(amd, s, 2 + s % 3, 200 + 40 * s, 128) for s in range(4)}
    wrong = []

    def work(t):
        for i in range(12):
            s = (t + i) % 4
            got, out = streams_of(amd, s, 2 + s % 3, 200 + 40 * s, 128)
            x = rows(s, 1, 64, 128)[0]
            q = quantize_per_channel(amd, x, 1, 1, 64, 128, 2, 32)
            if not all(np.array_equal(a, b) for a, b in zip(got, want[s][0])) or not np.array_equal(out, want[s][1]):
                wrong.append((t, i))
            del q

    threads = [threading.Thread(target=work, args=(t,)) for t in range(8)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not wrong


def test_kept_memory_is_bounded(amd):
    hip = C.CDLL("libamdhip64.so.7")

    def free_bytes():
        free, total = C.c_size_t(), C.c_size_t()
        assert hip.hipMemGetInfo(C.byref(free), C.byref(total)) == 0
        return free.value

    before = free_bytes()
    for tokens in (200_000, 700_000, 1_500_000, 400_000):  # up to ~3 GiB of arenas each
        c = KiviCache(amd, KiviConfig(8, 32, 32), 1, 8, 128)
        c.reserve(tokens)
        del c
    assert before - free_bytes() <= (1 << 30) + (64 << 20)


def test_allocating_calls_are_refused_under_capture(amd):
    hip = C.CDLL("libamdhip64.so.7")
    for _ in range(2):  # blocks of the sizes the captured call would take are in the pool
        c = KiviCache(amd, KiviConfig(2, 32, 32), 1, 2, 128)
        c.reserve(4096)
        del c
    c = KiviCache(amd, KiviConfig(2, 32, 32), 1, 2, 128)
    mem = DeviceArrays()
    n = 2 * 100 * 128
    k, v = rows(5, 2, 100, 128)
    dk, dv = mem.upload(k.reshape(-1)), mem.upload(v.reshape(-1))
    stream, graph = C.c_void_p(), C.c_void_p()
    assert hip.hipStreamCreate(C.byref(stream)) == 0
    assert hip.hipStreamBeginCapture(stream, 0) == 0  # global mode: hipMalloc is refused
    with pytest.raises(KiviError) as e:
        c.append_device(dk, n, dv, n, 100, stream.value)
    assert e.value.variant == "Device"
    hip.hipStreamEndCapture(stream, C.byref(graph))
    if graph:
        hip.hipGraphDestroy(graph)
    hip.hipGetLastError()
    assert c.sequence_length() == 0
    c.append(k, v, 100)  # and the cache still works
    assert c.sequence_length() == 100
    assert hip.hipStreamDestroy(stream) == 0
    mem.free()


class Capture:
    """A capture of the allocation-free attention on its own stream, begun by this thread; ``other`` runs
    on another thread before it ends."""

    def __init__(self, amd, mode):
        self.hip, self.mode, self.mem = C.CDLL("libamdhip64.so.7"), mode, DeviceArrays()
        self.cache = self.make(amd, 1)
        q = np.random.default_rng(3).standard_normal(4 * 128).astype(np.float32)
        self.n = q.size
        self.dq, self.out, self.out2 = self.mem.upload(q), self.mem.empty(q.size), self.mem.empty(q.size)
        self.streams = [C.c_void_p() for _ in range(2)]
        for s in self.streams:
            assert self.hip.hipStreamCreate(C.byref(s)) == 0
        self.cache.attention_device(self.dq, self.n, 4, 0.1, self.out2, self.n, self.streams[1].value)
        self.want = self.mem.download(self.out2, self.n)

    @staticmethod
    def make(amd, seed):
        c = KiviCache(amd, KiviConfig(2, 32, 32), 1, 2, 128)
        c.append(*rows(seed, 2, 300, 128), 300)
        return c

    def run(self, other):
        graph, failure = C.c_void_p(), []

        def work():
            try:
                other(self)
            except BaseException as e:  # reported by the test's own thread
                failure.append(e)

        assert self.hip.hipStreamBeginCapture(self.streams[0], self.mode) == 0
        self.cache.attention_device_noalloc(self.dq, self.n, 4, 0.1, self.out, self.n, self.streams[0].value)
        t = threading.Thread(target=work)
        t.start()
        t.join()
        rc = self.hip.hipStreamEndCapture(self.streams[0], C.byref(graph))
        self.hip.hipGetLastError()
        if failure:
            raise failure[0]
        return rc, graph


@pytest.mark.parametrize("mode", [1, 2])  # thread-local, relaxed
@pytest.mark.parametrize("what", ["cache", "growth", "session", "suffix", "quantized"])
def test_freeing_leaves_captures_of_other_threads_alone(amd, mode, what):
    cap = Capture(amd, mode)
    c = Capture.make(amd, 2)
    k, v = rows(9, 2, 1000, 128)
    dk, dv = cap.mem.upload(k.reshape(-1)), cap.mem.upload(v.reshape(-1))
    held = [None if what == "growth" else c if what == "cache" else c.share_prefix().session() if what == "session"
            else quantize_per_channel(amd, k[:, :992].copy(), 1, 2, 992, 128, 2, 32)]
    if what == "suffix":  # device rows on the default stream
        held[0] = c.share_prefix().session()
        held[0].append_device(dk, k.size, dv, v.size, 1000)
    if what == "cache":
        del c

    def other(cap):
        if what == "growth":
            c.append_device(dk, k.size, dv, v.size, 1000, cap.streams[1].value)
        held.clear()

    rc, graph = cap.run(other)
    assert rc == 0
    exe = C.c_void_p()
    assert cap.hip.hipGraphInstantiate(C.byref(exe), graph, None, None, C.c_size_t(0)) == 0
    for _ in range(3):
        assert cap.hip.hipMemcpy(C.c_void_p(cap.out), np.zeros(cap.n, np.float32).ctypes.data_as(C.c_void_p),
                                 C.c_size_t(4 * cap.n), 1) == 0
        assert cap.hip.hipGraphLaunch(exe, cap.streams[0]) == 0
        assert cap.hip.hipStreamSynchronize(cap.streams[0]) == 0
        assert np.array_equal(cap.mem.download(cap.out, cap.n), cap.want)
    assert cap.hip.hipGraphExecDestroy(exe) == 0 and cap.hip.hipGraphDestroy(graph) == 0
    for s in cap.streams:
        assert cap.hip.hipStreamDestroy(s) == 0
    cap.mem.free()


@pytest.mark.parametrize("replay", [False, True])
def test_a_buffer_waits_for_every_stream_that_reads_it(amd, replay):
    """Dense reconstructions on two streams, or by a graph's launch on another stream than it was captured
    on, then the cache freed at once and its buffers taken by the next one."""
    hip, mem = C.CDLL("libamdhip64.so.7"), DeviceArrays()
    units, n, dim = 8, 20000, 128
    cfg = KiviConfig(4, 32, 32)
    k, v = rows(11, units, n, dim)
    streams = [C.c_void_p() for _ in range(2)]
    for s in streams:
        assert hip.hipStreamCreateWithFlags(C.byref(s), 1) == 0  # non-blocking
    dk, dv = mem.upload(k.reshape(-1)), mem.upload(v.reshape(-1))
    outs = [(mem.alloc(k.size), mem.alloc(k.size)) for _ in streams]

    def filled():
        c = KiviCache(amd, cfg, 1, units, dim)
        c.reserve(n)
        return c

    c = filled()
    c.append(k, v, n)
    want = [np.asarray(x).view(np.uint32).copy() for x in c.dequantize()]
    for _ in range(4):
        if replay:
            graph, exe = C.c_void_p(), C.c_void_p()
            assert hip.hipStreamBeginCapture(streams[0], 1) == 0
            c.dequantize_device(outs[0][0], k.size, outs[0][1], k.size, streams[0].value)
            assert hip.hipStreamEndCapture(streams[0], C.byref(graph)) == 0
            assert hip.hipGraphInstantiate(C.byref(exe), graph, None, None, C.c_size_t(0)) == 0
            for _ in range(8):
                assert hip.hipGraphLaunch(exe, streams[1]) == 0
        else:
            for _ in range(8):
                for s, (a, b) in zip(streams, outs):
                    c.dequantize_device(a, k.size, b, k.size, s.value)
        del c
        c = filled()  # the same sizes: the buffers just given back
        c.append_device(dv, k.size, dk, k.size, n, streams[0].value)
        assert hip.hipDeviceSynchronize() == 0
        for a, b in outs[:1] if replay else outs:
            for ptr, x in ((a, want[0]), (b, want[1])):
                assert np.array_equal(mem.download(ptr, k.size).view(np.uint32), x.reshape(-1))
        if replay:
            assert hip.hipGraphExecDestroy(exe) == 0 and hip.hipGraphDestroy(graph) == 0
        del c
        c = filled()
        c.append(k, v, n)
    for s in streams:
        assert hip.hipStreamDestroy(s) == 0
    mem.free()


def test_a_buffer_waits_for_every_threads_own_stream(amd):
    """Dense reconstructions of two threads on hipStreamPerThread (one handle, a stream per thread), then
    the cache freed by a third and its buffers taken by the next one."""
    hip, mem = C.CDLL("libamdhip64.so.7"), DeviceArrays()
    units, n, dim, per_thread = 8, 20000, 128, 2
    cfg = KiviConfig(4, 32, 32)
    k, v = rows(11, units, n, dim)
    stream = C.c_void_p()
    assert hip.hipStreamCreateWithFlags(C.byref(stream), 1) == 0
    dk, dv = mem.upload(k.reshape(-1)), mem.upload(v.reshape(-1))
    outs = [(mem.alloc(k.size), mem.alloc(k.size)) for _ in range(2)]

    def filled():
        c = KiviCache(amd, cfg, 1, units, dim)
        c.reserve(n)
        return c

    for _ in range(4):
        c = filled()
        c.append(k, v, n)
        want = [np.asarray(x).view(np.uint32).copy() for x in c.dequantize()]
        held, queued, freed, failure = [c], threading.Barrier(3), threading.Event(), []
        del c

        def read(out):
            try:
                for _ in range(8):
                    held[0].dequantize_device(out[0], k.size, out[1], k.size, per_thread)
            except BaseException as e:
                failure.append(e)
            queued.wait(60)
            freed.wait(60)  # a thread's stream ends with the thread

        threads = [threading.Thread(target=read, args=(o,)) for o in outs]
        for t in threads:
            t.start()
        queued.wait(60)
        held.clear()
        c = filled()  # the same sizes: the buffers just given back
        c.append_device(dv, k.size, dk, k.size, n, stream.value)
        assert hip.hipDeviceSynchronize() == 0
        freed.set()
        for t in threads:
            t.join()
        assert not failure
        for out in outs:
            for ptr, x in zip(out, want):
                assert np.array_equal(mem.download(ptr, k.size).view(np.uint32), x.reshape(-1))
        del c
    assert hip.hipStreamDestroy(stream) == 0
    mem.free()


@pytest.mark.parametrize("how", ["one stream", "two streams", "graph", "growth"])
def test_a_suffix_waits_for_its_readers(amd, how):
    """Attention over a long suffix, then the session freed (or its suffix grown) at once and its buffers
    taken by the next session."""
    hip, mem = C.CDLL("libamdhip64.so.7"), DeviceArrays()
    units, n, dim = 2, 30000, 128
    prefix = Capture.make(amd, 4).share_prefix()
    k, v = rows(17, units, n, dim)
    dk, dv = mem.upload(k.reshape(-1)), mem.upload(v.reshape(-1))
    q = np.random.default_rng(5).standard_normal(4 * dim).astype(np.float32)
    dq = mem.upload(q)
    outs = [mem.empty(q.size) for _ in range(2)]
    streams = [C.c_void_p() for _ in range(3)]
    for s in streams:
        assert hip.hipStreamCreateWithFlags(C.byref(s), 1) == 0  # non-blocking

    def filled(stream):
        s = prefix.session()
        s.append_device(dk, k.size, dv, v.size, n, stream.value)
        assert hip.hipDeviceSynchronize() == 0
        return s

    def read(session, out, stream):
        kivi.sessions_attention_device(amd, [session], dq, q.size, 4, 0.1, out, q.size, stream.value)

    se = filled(streams[0])
    read(se, outs[0], streams[0])
    assert hip.hipDeviceSynchronize() == 0
    want = mem.download(outs[0], q.size)
    for _ in range(4):
        if how == "graph":
            graph, exe = C.c_void_p(), C.c_void_p()
            assert hip.hipStreamBeginCapture(streams[0], 1) == 0
            read(se, outs[0], streams[0])
            assert hip.hipStreamEndCapture(streams[0], C.byref(graph)) == 0
            assert hip.hipGraphInstantiate(C.byref(exe), graph, None, None, C.c_size_t(0)) == 0
            for _ in range(16):
                assert hip.hipGraphLaunch(exe, streams[1]) == 0
        else:
            for _ in range(16):
                read(se, outs[0], streams[0])
                if how == "two streams":
                    read(se, outs[1], streams[1])
        if how == "growth":
            se.append_device(dk, units * dim, dv, units * dim, 1, streams[0].value)
        else:
            del se
        se = prefix.session()
        se.append_device(dv, k.size, dk, k.size, n, streams[2].value)  # other rows, the same size
        assert hip.hipDeviceSynchronize() == 0
        for out in outs[:2 if how == "two streams" else 1]:
            assert np.array_equal(mem.download(out, q.size).view(np.uint32), want.view(np.uint32))
        if how == "graph":
            assert hip.hipGraphExecDestroy(exe) == 0 and hip.hipGraphDestroy(graph) == 0
        del se
        se = filled(streams[0])
        if how == "graph":  # sizes the new session's workspace
            read(se, outs[0], streams[0])
            assert hip.hipDeviceSynchronize() == 0
    del se
    for s in streams:
        assert hip.hipStreamDestroy(s) == 0
    mem.free()


@pytest.mark.parametrize("how", ["one stream", "two streams", "graph"])
def test_a_quantized_tensor_waits_for_its_readers(amd, how):
    """Reconstructions of a tensor, which is then freed at once and its buffers taken by the next one."""
    hip, mem = C.CDLL("libamdhip64.so.7"), DeviceArrays()
    units, n, dim = 8, 16384, 128
    x, y = rows(23, units, n, dim)
    dx, dy = mem.upload(x.reshape(-1)), mem.upload(y.reshape(-1))
    outs = [mem.alloc(x.size) for _ in range(2)]
    streams = [C.c_void_p() for _ in range(3)]
    for s in streams:
        assert hip.hipStreamCreateWithFlags(C.byref(s), 1) == 0  # non-blocking

    def make(data, stream):
        return kivi.quantize_device(amd, False, data, x.size, 1, units, n, dim, 4, 32, stream.value)

    t = make(dx, streams[0])
    want = np.asarray(t.dequantize()).view(np.uint32).reshape(-1).copy()
    for _ in range(4):
        if how == "graph":
            graph, exe = C.c_void_p(), C.c_void_p()
            assert hip.hipStreamBeginCapture(streams[0], 1) == 0
            t.dequantize_device(outs[0], x.size, streams[0].value)
            assert hip.hipStreamEndCapture(streams[0], C.byref(graph)) == 0
            assert hip.hipGraphInstantiate(C.byref(exe), graph, None, None, C.c_size_t(0)) == 0
            for _ in range(16):
                assert hip.hipGraphLaunch(exe, streams[1]) == 0
        else:
            for _ in range(16):
                t.dequantize_device(outs[0], x.size, streams[0].value)
                if how == "two streams":
                    t.dequantize_device(outs[1], x.size, streams[1].value)
        del t
        t = make(dy, streams[2])  # the buffers just given back
        assert hip.hipDeviceSynchronize() == 0
        for out in outs[:2 if how == "two streams" else 1]:
            assert np.array_equal(mem.download(out, x.size).view(np.uint32), want)
        if how == "graph":
            assert hip.hipGraphExecDestroy(exe) == 0 and hip.hipGraphDestroy(graph) == 0
        del t
        t = make(dx, streams[0])
        assert hip.hipDeviceSynchronize() == 0
    del t
    for s in streams:
        assert hip.hipStreamDestroy(s) == 0
    mem.free()


def test_a_tensor_may_outlive_its_stream(amd):
    """Readers queued on a stream that is destroyed (and perhaps its handle given to a new one) before the
    tensor is freed and its buffers taken by the next one. (Sessions free themselves the same way, but
    their prefix's batched calls need the previous call's stream.)"""
    hip, mem = C.CDLL("libamdhip64.so.7"), DeviceArrays()
    units, n, dim = 2, 32768, 128
    x, y = rows(29, units, n, dim)
    dx, dy = mem.upload(x.reshape(-1)), mem.upload(y.reshape(-1))
    out = mem.alloc(x.size)

    def stream():
        s = C.c_void_p()
        assert hip.hipStreamCreateWithFlags(C.byref(s), 1) == 0
        return s

    def make(data, s):
        return kivi.quantize_device(amd, False, data, x.size, 1, units, n, dim, 4, 32, s.value)

    want = None
    for _ in range(4):
        s = stream()
        t = make(dx, s)
        for _ in range(32):
            t.dequantize_device(out, x.size, s.value)
        if want is None:
            assert hip.hipStreamSynchronize(s) == 0
            want = mem.download(out, x.size)
        assert hip.hipStreamDestroy(s) == 0
        others = [stream() for _ in range(3)]
        del t
        t = make(dy, others[0])
        assert hip.hipDeviceSynchronize() == 0
        assert np.array_equal(mem.download(out, x.size).view(np.uint32), want.view(np.uint32))
        del t
        for s in others:
            assert hip.hipStreamDestroy(s) == 0
    mem.free()


@pytest.mark.parametrize("what", ["session", "quantized", "prefix"])
def test_a_refused_free_leaves_no_error_behind(amd, what):
    """An object freed while another thread captures in global mode (which refuses to free memory): the
    freeing thread's next call on another cache succeeds."""
    cap = Capture(amd, 0)
    k = rows(9, 2, 992, 128)[0]
    prefix = Capture.make(amd, 2).share_prefix()
    held = [prefix.session() if what == "session" else quantize_per_channel(amd, k, 1, 2, 992, 128, 2, 32)
            if what == "quantized" else prefix]
    del prefix

    def other(cap):
        held.clear()
        cap.cache.attention_device(cap.dq, cap.n, 4, 0.1, cap.out2, cap.n, cap.streams[1].value)

    assert np.array_equal(cap.mem.download(cap.out2, cap.n), cap.want)
    cap.run(other)  # global mode: the refusal may have ended the capture
    assert np.array_equal(cap.mem.download(cap.out2, cap.n), cap.want)
    for s in cap.streams:
        assert cap.hip.hipStreamDestroy(s) == 0
    cap.mem.free()


def free_device_bytes(hip):
    free, total = C.c_size_t(), C.c_size_t()
    assert hip.hipMemGetInfo(C.byref(free), C.byref(total)) == 0
    return free.value


def test_kept_memory_can_be_taken_back(amd):
    hip = C.CDLL("libamdhip64.so.7")
    kivi.release_pooled_memory(amd)
    assert kivi.release_pooled_memory(amd) == 0
    before = free_device_bytes(hip)
    c = KiviCache(amd, KiviConfig(8, 32, 32), 1, 8, 128)
    c.reserve(200_000)
    size = c.device_bytes()
    del c
    assert before - free_device_bytes(hip) >= size
    assert kivi.release_pooled_memory(amd) >= size
    assert before - free_device_bytes(hip) < size // 8


def test_scratch_gets_the_kept_memory(amd):
    """A host append whose staging fits the device only together with what the pool keeps."""
    hip, mem = C.CDLL("libamdhip64.so.7"), DeviceArrays()
    kivi.release_pooled_memory(amd)
    units, n, dim = 8, 80000, 128  # 328 MB of staging for the keys, as much for the values
    c = KiviCache(amd, KiviConfig(2, 32, 32), 1, units, dim)
    c.reserve(n)
    k = rows(21, units, n, dim)[0]
    big = KiviCache(amd, KiviConfig(8, 32, 32), 1, 8, 128)
    big.reserve(380_000)  # 973 MB
    mem.alloc((free_device_bytes(hip) - (280 << 20)) // 4)
    for _ in range(64):  # what was free rounds down: leave 200 to 232 MiB
        if free_device_bytes(hip) < 232 << 20:
            break
        mem.alloc(8 << 20)
    del big  # the pool's from here on
    try:
        c.append(k, k, n)
    finally:
        mem.free()
    assert c.sequence_length() == n


def test_a_block_past_the_bound_leaves_the_others(amd):
    """A tensor whose codes alone are above 1 GiB (1.5 GiB, with 96 MiB of parameters) freed after a small
    one (64 + 4 MiB): the codes go back to the device, the rest stays."""
    hip, mem = C.CDLL("libamdhip64.so.7"), DeviceArrays()
    kivi.release_pooled_memory(amd)
    n = 3 << 29
    data = mem.alloc(n)
    for elements in (1 << 26, n):
        q = kivi.quantize_device(amd, False, data, elements, 1, 1, elements // 128, 128, 8, 128)
        del q
    assert kivi.release_pooled_memory(amd) == (64 + 4 + 96) << 20
    assert hip.hipDeviceSynchronize() == 0
    mem.free()
