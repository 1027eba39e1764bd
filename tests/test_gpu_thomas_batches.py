"""GPU: the batched Thomas solves against the CPU checker bit for bit on both
sides of the rule that gives a batch to lanes or to waves, through the entry
point with host buffers and the one with device buffers, with arrays of the
systems' length and far longer ones, and with systems that are skipped."""
import numpy as np
import pytest

import oracle
from test_zz_no_alloc import device_solve, host_solve

pytestmark = pytest.mark.gpu


def batch(rng, lengths, spare=0):
    """Systems of the given lengths one after another (0: skipped), then
    `spare` rows that no system has."""
    lengths = np.asarray(lengths)
    off = np.concatenate([[0], np.cumsum(lengths)[:-1]]).astype(np.int32)
    n = int(lengths.sum()) + spare
    A, C = rng.uniform(-0.6, 0.4, n), rng.uniform(-0.6, 0.4, n)
    B = 1.0 + np.abs(A) + np.abs(C)
    B[1::2] *= -1.0
    return off, (lengths - 1).astype(np.int32), A, B, C, rng.normal(size=n), n


def mixed(rng, n, lo, hi, long=()):
    """n lengths in [lo, hi], a skipped system here and there, and a few long ones"""
    k = rng.integers(lo, hi + 1, n)
    k[rng.random(n) < 0.05] = 0
    for at, length in long:
        k[at] = length
    return k


BATCHES = {
    "1 of 1": (1, 1, 1, (), 0),
    "1 of 5": (1, 5, 5, (), 0),
    "1 of 6": (1, 6, 6, (), 0),
    "63 of 1-4": (63, 1, 4, (), 0),
    "64 of 1-4": (64, 1, 4, (), 0),
    "65 of 1-4": (65, 1, 4, (), 0),
    "64 of 5-6": (64, 5, 6, (), 0),
    "1000 of 1-7": (1000, 1, 7, (), 0),
    "1000 of 7-9": (1000, 7, 9, (), 0),
    "20000 of 2-40": (20000, 2, 40, (), 0),
    "20000 of 1-8 in long arrays": (20000, 1, 8, (), 800000),
    "130 of 1-5 in long arrays": (130, 1, 5, (), 5000),
    "one long among short": (1000, 1, 3, [(70, 900), (999, 600)], 0),
    "one long among short in long arrays": (1000, 1, 3, [(0, 511), (70, 900), (640, 6)], 100000),
}


@pytest.mark.parametrize("name", sorted(BATCHES))
def test_batches(name):
    n, lo, hi, long, spare = BATCHES[name]
    rng = np.random.default_rng(n + hi)
    lengths = mixed(rng, n, lo, hi, long)
    if n == 1:
        lengths[:] = lo
    args = batch(rng, lengths, spare)
    off, sn, A, B, C, D, _ = args
    want = np.full(A.size, -7.0)               # what skipped systems and spare rows keep
    for o, k in zip(off, lengths):
        if k:
            want[o:o + k] = oracle.thomas(A[o:o + k], B[o:o + k], C[o:o + k], D[o:o + k])
    for solve in (host_solve, device_solve):
        got = solve(*args)
        assert np.array_equal(got.view(np.int64), want.view(np.int64)), solve.__name__
