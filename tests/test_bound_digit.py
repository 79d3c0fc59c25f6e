"""The bounded selection's histogram buckets (bound_digit / bound_digit_edge, restated from their definition and run on the
host through the library's diagnostic export): monotone in the score key, and no value of a bucket or above lies below the
bucket's edge, for any row scale."""
import numpy as np
import pytest

from kernelswift_amd import _lib


def key(f):
    u = f.view(np.uint32).astype(np.uint64)
    u = np.where((u & 0x7FFFFFFF) == 0, 0, u)
    return np.where(u >> 31, ~u & 0xFFFFFFFF, u | 0x80000000)


def digit(f, M):
    u = f.view(np.uint32).astype(np.int64)
    m = u & 0x7FFFFFFF
    d = np.minimum(np.where(M > m, (M - m) >> 17, 0), 1023)
    return np.where(u >> 31, d, 2047 - d)


def edge(d, M):
    if d >= 1024:
        dd = 2047 - d
        low = (dd + 1) << 17
        return 0x80000000 | (M - low + 1 if dd < 1023 and M >= low else 0)
    return 1 if d == 0 else ~(0x80000000 | max(M - (d << 17), 0)) & 0xFFFFFFFF


def shipped(f, M):
    """The library's buckets of the values f and its 2048 edges."""
    f = np.ascontiguousarray(f, np.float32)
    d, e = np.empty(f.size, np.uint32), np.empty(2048, np.uint32)
    _lib.load().ks_dbg_bound_digits(f.ctypes.data, f.size, M, d.ctypes.data, e.ctypes.data)
    return d.astype(np.int64), e.astype(np.uint64)


@pytest.mark.parametrize("scale", [0.0, 1e-45, 1e-38, 2.0 ** -20, 0.3, 817.0, 2.0 ** 100, 3.4e38, np.inf])
def test_buckets_are_monotone_and_their_edges_bound_them(scale):
    g = np.random.default_rng(5)
    M = int(np.float32(scale).view(np.uint32))
    f = np.concatenate([g.standard_normal(20000) * 10.0 ** g.uniform(-44, 38, 20000), g.standard_normal(20000) * scale
                        if np.isfinite(scale) else [], [0.0, -0.0, np.inf, -np.inf, 3.4e38, -3.4e38, 1e-45, -1e-45]])
    f = f.astype(np.float32)
    k, (d, e) = key(f), shipped(f, M)
    np.testing.assert_array_equal(d, digit(f, M))
    np.testing.assert_array_equal(e, np.array([edge(b, M) for b in range(2048)], dtype=np.uint64))
    assert d.min() >= 0 and d.max() <= 2047
    o = np.lexsort((d, k))
    # -0 shares +0's key and may count in the bucket below it, which only lowers a threshold
    neg0 = f.view(np.uint32) == 0x80000000
    assert (np.diff(d[o][~neg0[o]]) >= 0).all()
    assert e.min() >= 1 and (np.diff(e.astype(np.int64)) >= 0).all()
    assert (k >= e[d]).all()
