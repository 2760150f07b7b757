"""Batched sessions of a shared prefix in groups of 16 rows (``-m gpu``).

Below 97 rows (sessions x query heads per KV head) the prefix's packed chunks run on the matrix
cores with the rows of all sessions as the columns of one tile, 16 at a time; from 97 on as a GEMM
over dequantized chunks. The cases sit at the edges: one row, a group less one, a whole group, one
more, the last count before the GEMM form and the first of it, head counts that do not divide 16,
a prefix batch above 1, prefixes without a packed chunk and with waves above a whole chunk,
sessions whose queries differ by six orders of magnitude (each row has its own operand range).

Every session against f64 attention over the dequantized prefix and its own suffix. Bar: the
matrix-core paths form products of 22 bits, 1e-4 at inputs of unit variance; a session whose
logits are scaled by s may be off by s times that of its largest value (first order in the logits).
"""

import numpy as np
import pytest

import kivi
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


@pytest.mark.parametrize("spread", [1.0, 1e6])
@pytest.mark.parametrize("case", CASES)
def test_rows_of_sessions_against_dense(amd, case, spread):
    bits, batch, heads, gq, n, count = case
    dim, qh = 128, heads * gq
    rng = np.random.default_rng(5100 + n + count)
    cache = KiviCache(amd, KiviConfig(bits, 32, 64), batch, heads, dim)
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
