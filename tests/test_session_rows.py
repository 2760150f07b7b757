"""Batched sessions of a shared prefix in groups of 16 rows (``-m gpu``).

Below 97 rows (sessions x query heads per KV head) and behind a short window the prefix's packed chunks
run on the matrix cores with the rows of all sessions as the columns of one tile, 16 at a time; from
97 on, or from 16 where that is faster, as a GEMM over dequantized chunks. The cases sit at the edges: one row, a group less one, a whole group, one
more, the last count before the GEMM form and the first of it, head counts that do not divide 16,
a prefix batch above 1, prefixes without a packed chunk and with waves above a whole chunk,
sessions whose queries differ by six orders of magnitude (each row has its own operand range).

Every session against f64 attention over the dequantized prefix and its own suffix. Bar: the
matrix-core paths form products of 22 bits, 1e-4 at inputs of unit variance; a session whose
logits are scaled by s may be off by s times that of its largest value (first order in the logits).
"""

import ctypes as C

import numpy as np
import pytest

import kivi
from helpers import DeviceArrays
from kivi import KiviCache, KiviConfig

pytestmark = pytest.mark.gpu

CASES = [
    # bits, batch, kv heads, query heads per KV head, prefix tokens, sessions
    (2, 1, 2, 1, 700, 1),
    (4, 1, 1, 3, 1000, 5),     # 15 rows
    (8, 2, 2, 2, 900, 8),      # 16 rows, batch 2
    (2, 1, 3, 1, 2500, 17),
    (4, 1, 2, 7, 1300, 6),     # 42 rows, eight-head windows
    (8, 1, 2, 8, 640, 12),     # 96 rows
    (2, 1, 1, 97, 0, 0),       # replaced below: 97 rows
    (2, 2, 1, 4, 100, 3),      # no packed keys beyond a residual: per-session attention
    (2, 1, 8, 4, 6100, 4),
]
CASES[6] = (2, 1, 2, 1, 1500, 64 + 33)  # 64 rows in a first launch group, 33 in the second
CASES.append((4, 1, 2, 2, 1500, 49))    # 98 rows: the GEMM form


# Other shapes: one launch for all sessions, each as its single-session launch. Lane splits, row splits
# alone (no packed chunk; a group of 8), the matrix-core chunks of other head_dims (with row splits
# behind them) and of groups of 64 (with window chunks), suffixes from empty to several splits.
OTHER = [
    # bits, group, dim, batch, kv heads, query heads per KV head, prefix tokens, sessions
    (4, 32, 96, 1, 2, 1, 900, 5),
    (2, 16, 80, 2, 1, 4, 1500, 3),
    (8, 16, 128, 1, 2, 7, 700, 66),     # two launch groups
    (2, 32, 128, 1, 2, 4, 20, 4),       # no packed keys
    (4, 8, 64, 1, 2, 3, 500, 3),
    (2, 32, 64, 1, 3, 4, 1300, 6),
    (4, 64, 256, 1, 1, 5, 800, 3),
    (8, 32, 192, 1, 1, 2, 640, 4),
    (2, 64, 128, 1, 2, 4, 1000, 5),
    (4, 128, 128, 2, 1, 8, 900, 3),
    (4, 8, 24, 1, 2, 3, 300, 3),        # generic splits: the sessions one by one
]


@pytest.mark.parametrize("case", OTHER)
def test_sessions_of_other_shapes_against_dense(amd, case):
    bits, group, dim, batch, heads, gq, n, count = case
    run(amd, bits, group, 2 * group, dim, batch, heads, gq, n, count, 1.0)


@pytest.mark.parametrize("spread", [1.0, 1e6])
@pytest.mark.parametrize("case", CASES)
def test_rows_of_sessions_against_dense(amd, case, spread):
    bits, batch, heads, gq, n, count = case
    run(amd, bits, 32, 64, 128, batch, heads, gq, n, count, spread)


# A long prefix window, which the row groups read once per session and the GEMM form once: the form
# is the one whose time is less, from 16 rows on.
WINDOWS = [
    # bits, residual, batch, kv heads, query heads per KV head, prefix tokens, sessions, GEMM form
    (8, 1024, 2, 8, 2, 1500, 24, True),    # 48 rows
    (4, 512, 1, 8, 1, 1200, 64, True),
    (2, 2048, 2, 8, 8, 2100, 2, False),    # 16 rows, no packed chunk behind the window
    (2, 1024, 4, 8, 1, 1100, 15, False),   # 15 rows
    (2, 1024, 4, 8, 1, 1100, 16, True),    # 16 rows
    (2, 1024, 4, 8, 1, 1050, 20, True),    # no packed chunk
    (4, 64, 2, 8, 4, 1500, 12, False),     # a short window
]


@pytest.mark.parametrize("case", WINDOWS)
def test_long_windows_run_once_for_all_rows(amd, case):
    bits, residual, batch, heads, gq, n, count, gemm = case
    kivi.timing_enable(amd)
    try:
        run(amd, bits, 32, residual, 128, batch, heads, gq, n, count, 1.0)
        assert (kivi.timing_read(amd, "attn_shared")[0] > 0) == gemm
    finally:
        kivi.timing_enable(amd, False)


@pytest.mark.parametrize("size", [1e-10, 1.0, 1e10])
@pytest.mark.parametrize("bits,gq,count,residual", [(2, 8, 3, 64), (4, 4, 6, 64), (8, 1, 20, 128)])
def test_value_magnitudes_keep_the_weights(amd, bits, gq, count, residual, size):
    """Values far from 1 cost no precision. Bar 5e-7 in relative 2-norm: a weight whose exponential
    takes in the values' power of two (2^33 and more) is rounded at 32 or above, 2^-19 / sqrt(3) * ln 2 =
    7.6e-7 rms; logits below 8 alone give 1e-7."""
    heads, dim, n = 4, 128, 1571
    rng = np.random.default_rng(5300 + bits)
    cache = KiviCache(amd, KiviConfig(bits, 32, residual), 1, heads, dim)
    k, v = (rng.standard_normal((heads, n, dim)).astype(np.float32) for _ in range(2))
    cache.append(k, v * np.float32(size), n)
    kd, vd = (x.reshape(heads, n, dim).astype(np.float64) for x in cache.dequantize())
    prefix = cache.share_prefix()
    sessions = [prefix.session() for _ in range(count)]
    q = rng.standard_normal((count, heads, gq, dim)).astype(np.float32)
    scale = np.float32(1 / np.sqrt(dim))
    got = kivi.sessions_attention(amd, sessions, q, heads * gq, scale).reshape(q.shape)
    logits = q.astype(np.float64) @ kd.swapaxes(-1, -2) * float(scale)
    w = np.exp(logits - logits.max(-1, keepdims=True))
    want = (w / w.sum(-1, keepdims=True)) @ vd
    assert np.linalg.norm(got - want) < 5e-7 * np.linalg.norm(want)


def run(amd, bits, group, residual, dim, batch, heads, gq, n, count, spread):
    qh = heads * gq
    rng = np.random.default_rng(5100 + n + count)
    cache = KiviCache(amd, KiviConfig(bits, group, residual), batch, heads, dim)
    k, v = (rng.standard_normal((batch, heads, n, dim)).astype(np.float32) for _ in range(2))
    cache.append(k, v, n)
    kd, vd = (x.reshape(batch, heads, n, dim).astype(np.float64) for x in cache.dequantize())
    prefix = cache.share_prefix()
    sessions, rows = [], []
    for i in range(count):
        m = (37 * i + 5) % 140
        s = prefix.session()
        ks, vs = (rng.standard_normal((batch, heads, m, dim)).astype(np.float32) for _ in range(2))
        s.append(ks, vs, m)
        sessions.append(s)
        rows.append((ks, vs))
    # with a spread, odd sessions' queries are that much smaller: their attention is near uniform
    size = np.where(np.arange(count) % 2 == 0, 1.0, 1.0 / spread).astype(np.float32)
    q = rng.standard_normal((count, batch, heads, gq, dim)).astype(np.float32) * size[:, None, None, None, None]
    scale = np.float32(1 / np.sqrt(dim))
    got = kivi.sessions_attention(amd, sessions, q, qh, scale).reshape(q.shape)
    for i in range(count):
        kk, vv = (np.concatenate([p, x.astype(np.float64)], 2) for p, x in zip((kd, vd), rows[i]))
        logits = q[i].astype(np.float64) @ kk.swapaxes(-1, -2) * float(scale)
        w = np.exp(logits - logits.max(-1, keepdims=True))
        want = (w / w.sum(-1, keepdims=True)) @ vv
        assert np.abs(got[i] - want).max() < 1e-4, f"session {i}"


def test_batch_captured_after_single_calls(amd):
    """Each session's own call has sized its workspace; a capture of all of them as one batch finds no
    workspace for a shared launch, runs them one by one and replays to the eager batch's rows."""
    hip = C.CDLL("libamdhip64.so.7")
    rng = np.random.default_rng(77)
    heads, gq, dim, n, count = 2, 2, 96, 900, 3
    qh, per = heads * gq, heads * gq * dim
    cache = KiviCache(amd, KiviConfig(4, 32, 64), 1, heads, dim)
    k, v = (rng.standard_normal((heads, n, dim)).astype(np.float32) for _ in range(2))
    cache.append(k, v, n)
    prefix = cache.share_prefix()
    sessions = [prefix.session() for _ in range(count)]
    mem = DeviceArrays()
    q = rng.standard_normal(count * per).astype(np.float32)
    dq, out = mem.upload(q), mem.empty(count * per)
    stream, graph, exe = C.c_void_p(), C.c_void_p(), C.c_void_p()
    assert hip.hipStreamCreate(C.byref(stream)) == 0

    def call(which, q_ptr, rows):
        kivi.sessions_attention_device(amd, which, q_ptr, rows, qh, 0.1, out, rows, stream.value)

    for s in sessions:
        call([s], dq, per)
    assert hip.hipStreamSynchronize(stream) == 0
    assert hip.hipStreamBeginCapture(stream, 0) == 0
    try:
        call(sessions, dq, count * per)
    finally:
        rc = hip.hipStreamEndCapture(stream, C.byref(graph))
    assert rc == 0
    assert hip.hipGraphInstantiate(C.byref(exe), graph, None, None, C.c_size_t(0)) == 0
    want = kivi.sessions_attention(amd, sessions, q, qh, 0.1)
    for _ in range(3):
        assert hip.hipMemcpy(C.c_void_p(out), np.zeros(count * per, np.float32).ctypes.data_as(C.c_void_p),
                             C.c_size_t(4 * count * per), 1) == 0
        assert hip.hipGraphLaunch(exe, stream) == 0
        assert hip.hipStreamSynchronize(stream) == 0
        got = mem.download(out, count * per)  # other splits than the batch's: twice the bar above
        assert np.abs(got - np.asarray(want).reshape(-1)).max() < 2e-4
    assert hip.hipGraphExecDestroy(exe) == 0 and hip.hipGraphDestroy(graph) == 0
    assert hip.hipStreamDestroy(stream) == 0
    mem.free()


@pytest.mark.parametrize("off", [0, 4])
@pytest.mark.parametrize("pinned", [False, True])
def test_suffix_rows_of_device_and_pinned_memory(amd, pinned, off):
    """Suffixes appended from this device's memory (a kernel's copy, or the copy engine 4 bytes off) and
    from pinned host memory (the copy engine): the rows of the host-pointer append."""
    hip, mem = C.CDLL("libamdhip64.so.7"), DeviceArrays()
    rng = np.random.default_rng(91)
    heads, dim = 3, 128
    cache = KiviCache(amd, KiviConfig(2, 32, 32), 1, heads, dim)
    k, v = (rng.standard_normal((heads, 100, dim)).astype(np.float32) for _ in range(2))
    cache.append(k, v, 100)
    prefix = cache.share_prefix()
    a, b = prefix.session(), prefix.session()
    for n in (5, 1, 40, 3):
        rows = [rng.standard_normal(heads * n * dim).astype(np.float32) for _ in range(2)]
        ptrs, hosts = [], []
        for x in rows:
            x = np.concatenate([np.zeros(off // 4, np.float32), x])
            if pinned:
                p = C.c_void_p()
                assert hip.hipHostMalloc(C.byref(p), C.c_size_t(x.nbytes), 0) == 0
                C.memmove(p, x.ctypes.data, x.nbytes)
                hosts.append(p)
                ptrs.append(p.value + off)
            else:
                ptrs.append(mem.upload(x) + off)
        a.append_device(ptrs[0], rows[0].size, ptrs[1], rows[1].size, n)
        b.append(rows[0], rows[1], n)
        assert hip.hipDeviceSynchronize() == 0
        for p in hosts:
            assert hip.hipHostFree(p) == 0
    q = rng.standard_normal(2 * heads * dim).astype(np.float32)
    assert np.array_equal(a.attention(q, 2 * heads, 0.1), b.attention(q, 2 * heads, 0.1))
    mem.free()
