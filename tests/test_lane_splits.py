"""Attention of the shapes the matrix-core kernels do not take (``-m gpu``): head_dims that are
multiples of 16 but not 64, 128, 192 or 256, and groups that are multiples of 16 but neither 32 nor
multiples of 64.

Their packed chunks run as lane splits (up to 16 chunks each, 1, 2 or 4 query heads per workgroup),
so the cases sit at the edges of that form: one chunk, splits of 4, 5, 8, 9, 16 and more chunks,
lanes per token (head_dim / 16) that do and do not divide a wave, every code width, odd numbers of
heads, a group of 48 tokens. Against the oracle within the parity tolerance, and against f64
attention over the dequantized cache: the kernel reconstructs every element as the reference does
and sums products in f32, eight in a row, two such sums, then at most 18 partial sums in a row (15, or
16 in each of four chains from head_dim 256 on), so its outputs lie within (16 + 12) 2^-24 of the products' magnitude sum, 1.7e-6 of a logit's; 2e-5 absolute bounds that at
these inputs (logits below 2^4 in magnitude sum, values below 2^3)."""

import numpy as np
import pytest

from kivi import KiviCache, KiviConfig, KiviError
from helpers import DeviceArrays
from test_parity import assert_close

pytestmark = pytest.mark.gpu

def dense_attention(cache, q, heads, scale):
    """f64 attention of q [batch, heads, gq, dim] over the cache's dequantized rows."""
    batch, _, _, dim = q.shape
    kd, vd = (x.reshape(batch, heads, -1, dim).astype(np.float64) for x in cache.dequantize())
    logits = q.astype(np.float64) @ kd.swapaxes(-1, -2) * float(scale)
    w = np.exp(logits - logits.max(-1, keepdims=True))
    return (w / w.sum(-1, keepdims=True)) @ vd


# Grids the split planner evens out (matrix-core kernels): a few workgroups above 256, waves just
# above a whole chunk. Bar of the matrix-core path against f64 (22-bit products): 1e-4.
UNEVEN = [
    # bits, group, dim, batch, kv heads, query heads per KV head, tokens
    (2, 32, 64, 5, 8, 4, 2000),    # 40 units x 29 chunks: 7 splits of 2 chunks per wave -> 8 of 1
    (4, 64, 256, 7, 8, 1, 700),    # 56 units x 9 chunks
    (8, 32, 128, 5, 8, 3, 2500),
    (4, 32, 128, 3, 8, 7, 3000),   # eight-head kernel
]


@pytest.mark.parametrize("case", UNEVEN)
def test_evened_grids_against_dense(amd, case):
    bits, group, dim, batch, heads, gq, n = case
    rng = np.random.default_rng(4700 + n)
    a = KiviCache(amd, KiviConfig(bits, group, 128), batch, heads, dim)
    k, v = (rng.standard_normal((batch, heads, n, dim)).astype(np.float32) for _ in range(2))
    q = rng.standard_normal((batch, heads, gq, dim)).astype(np.float32)
    a.append(k, v, n)
    scale = np.float32(1 / np.sqrt(dim))
    got = a.attention(q, heads * gq, scale).reshape(q.shape)
    assert np.abs(got - dense_attention(a, q, heads, scale)).max() < 1e-4


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
    assert np.abs(got - dense_attention(a, q.reshape(got.shape), heads, scale)).max() < 2e-5
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


@pytest.mark.parametrize("bits,group,residual", [(4, 16, 32), (8, 16, 256), (4, 8, 16)])
def test_wide_heads_sum_in_short_chains(amd, bits, group, residual):
    """head_dim 1024, lane splits and row splits: the 64 partial sums of a logit in four chains of 16, not
    one of 64, which rounds twice as much in the rms. Relative 2-norm off f64 attention, rms of eight
    caches: one chain 3.1e-7 to 3.4e-7, four 2.0e-7 (the rest of it is the softmax's and the mix's)."""
    units, gq, n, dim = 2, 4, 300, 1024
    errors = []
    for seed in range(8):
        rng = np.random.default_rng(5400 + seed)
        k, v = (rng.standard_normal((1, units, n, dim)).astype(np.float32) for _ in range(2))
        k[..., 0] *= 10
        c = KiviCache(amd, KiviConfig(bits, group, residual), 1, units, dim)
        c.append(k, v, n)
        q = rng.standard_normal((1, units, gq, dim)).astype(np.float32)
        scale = np.float32(1 / np.sqrt(dim))
        want = dense_attention(c, q, units, scale)
        got = c.attention(q, units * gq, scale).reshape(q.shape)
        errors.append(np.linalg.norm(got - want) / np.linalg.norm(want))
    assert np.sqrt(np.mean(np.square(errors))) < 2.6e-7
