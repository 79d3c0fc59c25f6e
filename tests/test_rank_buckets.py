"""The rank store's buckets (ks::RankScale, run on the host through the library's diagnostic export): monotone in the score
key over any range, infinities and the largest finite values among the keys and as the range's ends."""
import numpy as np
import pytest

from kernelswift_amd import _lib

FMAX = np.float32(3.4028235e38)
TINY = np.float32(1e-45)


def key(f):
    u = np.asarray(f, np.float32).view(np.uint32)
    u = np.where((u & 0x7FFFFFFF) == 0, np.uint32(0), u)
    return np.where(u >> 31, ~u, u | np.uint32(0x80000000)).astype(np.uint32)


def buckets(keys, kmin, kmax):
    keys = np.ascontiguousarray(keys, np.uint32)
    out = np.empty_like(keys)
    _lib.load().ks_dbg_rank_buckets(keys.ctypes.data, keys.size, int(kmin), int(kmax), out.ctypes.data)
    return out


@pytest.mark.parametrize("lo,hi", [(-np.inf, 2.0), (-3.0, np.inf), (-np.inf, np.inf), (-FMAX, FMAX), (-FMAX, -1e38),
                                   (0.0, FMAX), (1.0, 2.0), (1.0, 1.0), (-5.0, 3.0), (-np.inf, -np.inf), (np.inf, np.inf),
                                   (-TINY, TINY), (0.0, 0.0), (1e30, np.inf), (-1e-38, 1e-38)])
def test_rank_buckets_are_monotone(lo, hi):
    g = np.random.default_rng(3)
    lo, hi = np.float32(lo), np.float32(hi)
    with np.errstate(over="ignore"):
        f = (g.standard_normal(6000) * 10.0 ** g.uniform(-45, 39, 6000)).astype(np.float32)
    f = np.concatenate([f, np.float32([lo, hi, 0.0, 1.0, -1.0, 2.0, -3.0, 5.0, FMAX, -FMAX, np.inf, -np.inf, TINY, -TINY])])
    f = f[(f >= lo) & (f <= hi)]
    k = np.sort(key(f))
    for kmin in (key(lo), np.uint32(1)):  # the smallest key, or an end below every value
        b = buckets(k, kmin, key(hi)).astype(np.int64)
        assert (np.diff(b) >= 0).all() and b.min() >= 0 and b.max() <= 2047


def test_rank_buckets_use_their_range():
    # the largest value alone does not take the whole range's resolution with it
    k = key(np.linspace(-4.0, 3.0, 1000, dtype=np.float32))
    assert np.unique(buckets(k, k[0], k[-1])).size > 700
    k = key(np.float32([-np.inf, -3.0, 0.0, 5.0]))
    b = buckets(k, k[0], k[-1])
    assert b[0] == 0 and b[1] > 0
