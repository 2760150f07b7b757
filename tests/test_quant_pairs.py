"""Quantizers of head_dims other than 64, 128 and 256, and of groups those do not take (``-m gpu``).

A lane holds two channels there, and a workgroup's lanes run over (run of tokens, channel pair)
items, so the cases sit at that form's edges: the narrowest heads, head_dims whose pairs do not
divide a workgroup, more than 256 items per value block, the last items of a unit, groups of 16, 32,
64 and 128 (keys of 128 are read twice), blocks that fill across appends and from the ring, inputs 4
bytes off (the general kernels). Every stream, the standalone codec's too, bit for bit against the
oracle, with planted zero minima of either sign, constant groups and infinities (a group that spans
one gets codes 0)."""

import numpy as np
import pytest

import kivi
from kivi import KiviCache, KiviConfig, quantize_per_channel, quantize_per_token
from helpers import DeviceArrays, signed_zero_rows

pytestmark = pytest.mark.gpu

CASES = [
    # bits, group, dim, units
    (2, 16, 16, 3), (2, 16, 80, 2), (2, 32, 96, 3), (4, 16, 48, 2), (4, 32, 160, 2), (4, 64, 192, 1),
    (4, 32, 96, 2), (8, 16, 112, 2), (8, 32, 96, 3), (8, 64, 320, 1), (2, 64, 256, 1), (2, 128, 128, 2),
    (4, 128, 256, 1), (8, 128, 384, 1), (8, 16, 512, 1), (4, 16, 1024, 1),
]


def rows(rng, shape, group):
    x = rng.standard_normal(shape).astype(np.float32)
    x[0] = signed_zero_rows(rng, shape[1:])       # zero minima of both signs
    x[-1, : 2 * group, : shape[2] // 2] = 1.25    # constant groups on both axes
    x[-1, shape[1] // 2, 0] = np.inf
    return x


def same(a, b):
    return np.array_equal(np.asarray(a).view(np.uint32), np.asarray(b).view(np.uint32))


@pytest.mark.parametrize("case", CASES)
def test_cache_streams_match_oracle(amd, oracle, case):
    bits, group, dim, units = case
    rng = np.random.default_rng(6200 + dim + bits)
    cfg = KiviConfig(bits, group, 2 * group)
    a, o = KiviCache(amd, cfg, 1, units, dim), KiviCache(oracle, cfg, 1, units, dim)
    for n in (2 * group + 1, 3, 5 * group + 7, 2 * group - 1, 70):
        k, v = rows(rng, (units, n, dim), group), rows(rng, (units, n, dim), group)
        a.append(k, v, n)
        o.append(k, v, n)
    for got, want, name in zip(a.export_streams(), o.export_streams(), ("key codes", "key params", "value codes", "value params")):
        assert same(got, want), name


@pytest.mark.parametrize("off", [0, 4])
@pytest.mark.parametrize("case", CASES)
def test_codec_matches_oracle(amd, oracle, case, off):
    bits, group, dim, units = case
    rng = np.random.default_rng(6300 + dim + bits)
    n = 3 * group
    data = rows(rng, (units, n, dim), group)
    mem = DeviceArrays()
    try:
        ptr = mem.upload(np.concatenate([np.zeros(off // 4, np.float32), data.reshape(-1)])) + off
        for per_channel in (True, False):
            want = (quantize_per_channel if per_channel else quantize_per_token)(oracle, data, 1, units, n, dim, bits, group)
            got = kivi.quantize_device(amd, per_channel, ptr, data.size, 1, units, n, dim, bits, group)
            assert same(got.codes(), want.codes()) and same(got.scale_zero(), want.scale_zero())
    finally:
        mem.free()


@pytest.mark.parametrize("bits,group,dim", [
    (8, 4, 4), (4, 8, 24), (2, 16, 16), (2, 16, 80), (4, 32, 96), (8, 16, 112), (4, 64, 320), (8, 16, 1024), (2, 64, 1024)])
def test_single_token_appends_match_oracle(amd, oracle, bits, group, dim):
    """One-launch appends (copy, eviction, window write) of head_dims that are no whole waves and of
    the widest, across a window's fill, evictions and key flushes."""
    rng = np.random.default_rng(6400 + dim)
    cfg, units = KiviConfig(bits, group, group), 2
    a, o = KiviCache(amd, cfg, 1, units, dim), KiviCache(oracle, cfg, 1, units, dim)
    for step in range(3 * group + 70):
        k, v = rows(rng, (units, 1, dim), 0), rows(rng, (units, 1, dim), 0)
        k[np.isinf(k)] = 0
        v[np.isinf(v)] = np.inf if step == 7 else 0
        a.append(k, v, 1)
        o.append(k, v, 1)
    for got, want, name in zip(a.export_streams(), o.export_streams(), ("key codes", "key params", "value codes", "value params")):
        assert same(got, want), name
    for got, want in zip(a.dequantize(), o.dequantize()):
        assert same(got[~np.isnan(want)], want[~np.isnan(want)])


# pair forms and one-launch appends at head_dims the wave forms do not take
NAN_CASES = [(2, 16, 80), (4, 32, 96), (8, 16, 112), (4, 64, 320), (8, 128, 384), (2, 16, 1024)]


def nan_rows(rng, shape, group):
    """Single NaNs, whole channel groups of NaNs in some rows, and NaN-only channels over many rows."""
    x = rng.standard_normal(shape).astype(np.float32)
    flat = x.reshape(-1)
    flat[rng.choice(flat.size, max(1, flat.size // 50), replace=False)] = np.nan
    x[0, shape[1] // 3, :group] = np.nan
    x[-1, -1, -group:] = np.nan
    x[-1, :, 3] = np.nan
    return x


def same_or_nan(a, b):
    a, b = np.asarray(a), np.asarray(b)
    if a.dtype != np.float32:
        return np.array_equal(a, b)
    return np.array_equal(np.isnan(a), np.isnan(b)) and same(a[~np.isnan(a)], b[~np.isnan(b)])


def check_streams(a, o):
    for got, want, name in zip(a.export_streams(), o.export_streams(), ("key codes", "key params", "value codes", "value params")):
        assert same_or_nan(got, want), name


@pytest.mark.parametrize("bits,group,dim", NAN_CASES)
def test_nans_are_passed_over(amd, oracle, bits, group, dim):
    """A NaN takes no part in a group's minimum and maximum and gets code 0; a group of NaNs alone keeps
    the reduction's initial values, zero +inf and scale -inf (src/quant.rs:303, 356: f32::min / max).
    Long appends, the standalone codec, and the same rows token by token."""
    rng = np.random.default_rng(6500 + dim)
    cfg, units, n = KiviConfig(bits, group, group), 2, 4 * group
    k, v = nan_rows(rng, (units, n, dim), group), nan_rows(rng, (units, n, dim), group)
    a, o = KiviCache(amd, cfg, 1, units, dim), KiviCache(oracle, cfg, 1, units, dim)
    for c in (a, o):
        c.append(k, v, n)
    check_streams(a, o)
    for fn in (quantize_per_channel, quantize_per_token):
        got, want = (fn(x, k, 1, units, n, dim, bits, group) for x in (amd, oracle))
        assert same_or_nan(got.codes(), want.codes()) and same_or_nan(got.scale_zero(), want.scale_zero())
    steps = min(n, 160)
    a, o = KiviCache(amd, cfg, 1, units, dim), KiviCache(oracle, cfg, 1, units, dim)
    for t in range(steps):
        for c in (a, o):
            c.append(np.ascontiguousarray(k[:, n - steps + t:n - steps + t + 1]),
                     np.ascontiguousarray(v[:, n - steps + t:n - steps + t + 1]), 1)
    for t in range(group):  # evict them all
        for c in (a, o):
            c.append(np.ones((units, 1, dim), np.float32), np.ones((units, 1, dim), np.float32), 1)
    check_streams(a, o)
