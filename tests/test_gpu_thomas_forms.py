"""GPU: the speculative batched Thomas against the CPU checker bit for bit
where its forms change: system lengths around the one-lane limit and the
powers of two of its rows per lane, chunk boundaries, and values that leave
the range of its shared reciprocals (signed zeros, tiny and huge entries,
zero pivots, infinities and NaN)."""
import numpy as np
import pytest

import oracle
from hydist_amd._lib import thomas_batch

pytestmark = pytest.mark.gpu


def system(rng, n):
    A, C = rng.uniform(-0.6, 0.4, n), rng.uniform(-0.6, 0.4, n)
    B = 1.0 + np.abs(A) + np.abs(C)
    B[1::2] *= -1.0
    return [A, B, C, rng.normal(size=n)]


def same(x, y):
    nan = np.isnan(x) & np.isnan(y)
    return np.array_equal(x.view(np.int64)[~nan], y.view(np.int64)[~nan])


@pytest.mark.parametrize("spec", [True, False])
def test_lengths(spec):
    rng = np.random.default_rng(5)
    edges = [1, 2, 3, 4, 33, 34, 35, 65, 66, 67, 129, 130, 131, 257, 258, 259, 510, 511, 512, 513, 1021, 1022, 1100]
    systems = [system(rng, n) for n in edges]
    for x, s in zip(thomas_batch(systems, spec=spec), systems):
        assert same(x, oracle.thomas(*s)), len(x)


@pytest.mark.parametrize("case", ["zero_rhs", "minus_zero_rhs", "minus_zero_upper", "zero_upper", "tiny_rhs",
                                  "denormal_rhs", "tiny_upper", "huge_rhs", "huge_rows", "zero_pivot", "inf", "nan"])
@pytest.mark.parametrize("n", [20, 100, 240, 500])
def test_values_outside_the_reciprocal_range(case, n):
    rng = np.random.default_rng(n)
    systems = []
    for _ in range(6):
        s = system(rng, n)
        A, B, C, D = s
        k = int(rng.integers(2, n - 2))
        if case == "zero_rhs":
            D[k:] = 0.0
        elif case == "minus_zero_rhs":
            D[:] = -0.0
        elif case == "minus_zero_upper":
            C[::3] = -0.0
        elif case == "zero_upper":
            C[::3] = 0.0
        elif case == "tiny_rhs":
            D *= 1e-250
        elif case == "denormal_rhs":
            D *= 1e-310
        elif case == "tiny_upper":
            C[k] = 1e-260
        elif case == "huge_rhs":
            D[k] = 1e300
        elif case == "huge_rows":
            for a in (A, B, C, D):
                a *= 1e100
        elif case == "zero_pivot":
            A[k] = B[k] = 0.0
        elif case == "inf":
            D[k] = np.inf
        else:
            D[k] = np.nan
        systems.append(s)
    for x, s in zip(thomas_batch(systems, spec=True), systems):
        assert same(x, oracle.thomas(*s)), case
