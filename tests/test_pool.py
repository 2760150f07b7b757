"""Device memory the library keeps between objects (``-m gpu``): a buffer given back and taken again
holds nothing of its previous owner, threads and streams share the pool, what it keeps is bounded,
and a call that would allocate is refused under stream capture as hipMalloc would be."""

import ctypes as C
import threading

import numpy as np
import pytest

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
