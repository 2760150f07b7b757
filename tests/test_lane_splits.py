"""Attention of the shapes the matrix-core kernels do not take (``-m gpu``): head_dims that are
multiples of 16 but not 64, 128, 192 or 256, and groups that are multiples of 16 but neither 32 nor
multiples of 64.

Their packed chunks run as lane splits (up to 16 chunks each, 1, 2 or 4 query heads per workgroup),
so the cases sit at the edges of that form: one chunk, splits of 4, 5, 8, 9, 16 and more chunks,
lanes per token (head_dim / 16) that do and do not divide a wave, every code width, odd numbers of
heads, a group of 48 tokens. Against the oracle within the parity tolerance, and against f64
attention over the dequantized cache: the kernel reconstructs every element as the reference does
and sums products in f32, at most 16 in a row before a tree, so its outputs lie within
(16 + 12) 2^-24 of the products' magnitude sum, 1.7e-6 of a logit's; 2e-5 absolute bounds that at
these inputs (logits below 2^4 in magnitude sum, values below 2^3)."""

import numpy as np
import pytest

from kivi import KiviCache, KiviConfig, KiviError
from helpers import DeviceArrays
from test_parity import assert_close

pytestmark = pytest.mark.gpu

CASES = [
    # bits, group, residual, dim, batch, kv heads, query heads per KV head, tokens
    (2, 32, 32, 32, 1, 1, 1, 96),          # one packed chunk
    (4, 16, 16, 80, 1, 2, 1, 64 * 4 + 16),
    (8, 16, 32, 16, 2, 1, 2, 64 * 5 + 40),  # one lane per token
    (2, 16, 16, 64, 1, 3, 3, 64 * 8 + 17),
    (4, 32, 64, 96, 1, 2, 4, 64 * 9 + 65),
    (8, 32, 32, 160, 1, 1, 5, 700),
    (2, 48, 96, 48, 2, 2, 9, 1300),
    (4, 16, 128, 128, 1, 2, 16, 1111),
    (8, 16, 16, 256, 1, 1, 7, 500),
    (8, 32, 32, 1024, 1, 1, 2, 333),       # the widest heads: a wave per token
    (2, 32, 96, 96, 40, 8, 1, 64 * 33 + 1),  # splits of 16 chunks (enough workgroups without shorter ones)
    (4, 16, 32, 112, 40, 8, 2, 64 * 18 + 50),  # splits of 9 chunks
]


@pytest.mark.parametrize("case", CASES)
def test_lane_splits_against_oracle_and_dense(amd, oracle, case):
    bits, group, residual, dim, batch, heads, gq, n = case
    rng = np.random.default_rng(4100 + n)
    cfg, qh, scale = KiviConfig(bits, group, residual), heads * gq, np.float32(1 / np.sqrt(dim))
    k = rng.standard_normal((batch, heads, n, dim)).astype(np.float32)
    v = rng.standard_normal((batch, heads, n, dim)).astype(np.float32)
    q = rng.standard_normal((batch, qh, dim)).astype(np.float32)
    a = KiviCache(amd, cfg, batch, heads, dim)
    a.append(k, v, n)
    got = a.attention(q, qh, scale).reshape(batch, heads, gq, dim)
    kd, vd = (x.reshape(batch, heads, n, dim).astype(np.float64) for x in a.dequantize())
    logits = q.reshape(batch, heads, gq, dim).astype(np.float64) @ kd.swapaxes(-1, -2) * float(scale)
    w = np.exp(logits - logits.max(-1, keepdims=True))
    dense = (w / w.sum(-1, keepdims=True)) @ vd
    assert np.abs(got - dense).max() < 2e-5
    if batch * heads < 10:
        o = KiviCache(oracle, cfg, batch, heads, dim)
        o.append(k, v, n)
        assert_close(got.reshape(-1), o.attention(q, qh, scale))
    # the allocation-free entry point: the same bits, or Capacity beyond its workspace
    mem = DeviceArrays()
    try:
        dq, out = mem.upload(q.reshape(-1)), mem.empty(q.size)
        try:
            a.attention_device_noalloc(dq, q.size, qh, scale, out, q.size)
        except KiviError as e:
            assert e.variant == "Capacity" and e.a > 2 << 20
        else:
            assert np.array_equal(mem.download(out, q.size), got.reshape(-1))
    finally:
        mem.free()
