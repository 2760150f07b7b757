"""Attention whose split plan meets a limit (``-m gpu``): partials around the 2,097,152 floats of the
static workspace, and head counts whose generic splits are bounded by LDS.

Each case against f64 attention over the dequantized cache, and the allocation-free entry point
against the allocating one: the same bits, or Capacity where the counted partials (stated per case)
exceed the workspace. Bars: the f32 kernels sum up to 16 products in a row before a tree (2e-5 at
inputs of unit variance, see test_lane_splits.py); generic splits sum a head's dim products in one
chain and a split's up to 256 weighted values in another, (256 + 24) 2^-24 of a magnitude sum below
2^3: 1.4e-4; the matrix-core path 1e-4."""

import numpy as np
import pytest

from kivi import KiviCache, KiviConfig, KiviError
from helpers import DeviceArrays
from test_lane_splits import dense_attention

pytestmark = pytest.mark.gpu

STATIC_FLOATS = 2 << 20


def check(amd, bits, group, residual, dim, units, gq, n, bar, counted):
    rng = np.random.default_rng(8800 + n)
    scale, qh = np.float32(1 / np.sqrt(dim)), gq
    cache = KiviCache(amd, KiviConfig(bits, group, residual), units, 1, dim)
    k, v = (rng.standard_normal((units, 1, n, dim), dtype=np.float32) for _ in range(2))
    cache.append(k, v, n)
    q = rng.standard_normal((units, 1, gq, dim), dtype=np.float32)
    got = cache.attention(q.reshape(-1), qh, scale)
    assert np.abs(got.reshape(q.shape) - dense_attention(cache, q, 1, scale)).max() < bar
    mem = DeviceArrays()
    try:
        dq, out = mem.upload(q.reshape(-1)), mem.empty(q.size)
        if counted > STATIC_FLOATS:
            with pytest.raises(KiviError) as e:
                cache.attention_device_noalloc(dq, q.size, qh, scale, out, q.size)
            assert (e.value.variant, e.value.a, e.value.b) == ("Capacity", counted, STATIC_FLOATS)
        else:
            cache.attention_device_noalloc(dq, q.size, qh, scale, out, q.size)
            assert np.array_equal(mem.download(out, q.size).view(np.uint32), got.view(np.uint32))
    finally:
        mem.free()


GENERIC = [
    # bits, group, dim, units, query heads per KV head, tokens, counted partials
    (4, 8, 24, 16, 64, 10500, 16 * 83 * 64 * 26),   # splits of 128: 38,912 bytes of LDS
    (4, 8, 24, 1, 160, 20000, 625 * 160 * 26),      # splits of 32: 35,840 bytes
    (8, 4, 8, 1, 256, 40000, 1250 * 256 * 10),      # splits of 32: 40,960 bytes
    (8, 4, 8, 1, 1024, 500, 16 * 1024 * 10),        # all of a CU's LDS
    (4, 8, 24, 3, 100, 3000, 3 * 47 * 100 * 26),    # fits the static workspace
]


@pytest.mark.parametrize("bits,group,dim,units,gq,n,counted", GENERIC)
def test_generic_splits_of_many_heads(amd, bits, group, dim, units, gq, n, counted):
    check(amd, bits, group, 2 * group, dim, units, gq, n, 1.4e-4, counted)


AROUND_STATIC = [
    # bits, group, residual, dim, units, query heads per KV head, tokens, bar, counted partials
    (4, 64, 64, 256, 340, 4, 447, 1e-4, 340 * 5 * 4 * 258),   # an evened grid and its row splits
    (4, 8, 32, 1024, 8, 4, 1200, 2e-5, 8 * 5 * 4 * 1026),     # row splits alone
    (4, 16, 1024, 1024, 8, 4, 1500, 2e-5, 8 * 6 * 4 * 1026),  # lane splits before a long window
    (4, 16, 16, 48, 1000, 32, 200, 2e-5, 1000 * 32 * 50),     # only the counted plan fits
    (4, 8, 16, 48, 130, 12, 10000, 2e-5, 130 * 40 * 12 * 50),  # counted too large: the usual plan
]


@pytest.mark.parametrize("bits,group,residual,dim,units,gq,n,bar,counted", AROUND_STATIC)
def test_plans_around_the_static_workspace(amd, bits, group, residual, dim, units, gq, n, bar, counted):
    """Cases whose usual plan takes more partials than the static workspace holds."""
    check(amd, bits, group, residual, dim, units, gq, n, bar, counted)
