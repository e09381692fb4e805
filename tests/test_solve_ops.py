"""The superposition solve's short square root, reciprocal and division
(gta_kabsch.h) against numpy's correctly rounded float32 operators, bit for bit
over the ranges that the solve uses: results that are bit-identical to the
plain operators' rest on it."""
import numpy as np
import pytest

from gtalign_alpha_amd.batch import GtaBatch
from gtalign_alpha_amd.capi import default_options

pytestmark = pytest.mark.gpu
SQRT, RCP, DIV = 0, 1, 2


@pytest.fixture(scope="module")
def b():
    with GtaBatch(0, default_options(), max_qrys=1, max_qry_poss=8, max_refs=1, max_ref_poss=8) as bt:
        yield bt


def mantissas(exponent):
    """Every float32 in [2^exponent, 2^(exponent + 1))."""
    return (np.arange(1 << 23, dtype=np.uint32) | np.uint32((exponent + 127) << 23)).view(np.float32)


def bits(x):
    return x.view(np.uint32)


@pytest.mark.parametrize("exponent", [0, 1, -100, 101])
def test_square_root(b, exponent):
    x = mantissas(exponent)
    assert np.array_equal(bits(b.solve_op(SQRT, x)), bits(np.sqrt(x)))


@pytest.mark.parametrize("exponent", [0, -60, 60])
def test_reciprocal(b, exponent):
    x = mantissas(exponent)
    assert np.array_equal(bits(b.solve_op(RCP, x)), bits(np.float32(1) / x))


def edges():
    p = np.exp2(np.arange(-40, 41, dtype=np.float64)).astype(np.float32)
    return np.concatenate([p, np.nextafter(p, np.float32(0)), np.nextafter(p, np.float32(np.inf))])


def test_division(b):
    """Divisors are counts or mean magnitudes (1e-18 to 1e18); numerators of
    either sign from 2^-100 to 9 times the divisor, whole and half ulps apart."""
    rng = np.random.default_rng(7)
    n = 1 << 23
    d = np.exp(rng.uniform(np.log(1e-18), np.log(1e18), n)).astype(np.float32)
    d[: n // 4] = rng.integers(1, 65536, n // 4)                    # counts
    ratio = np.exp(rng.uniform(np.log(1e-9), np.log(9.0), n)) * rng.choice([-1.0, 1.0], n)
    a = (d * ratio).astype(np.float32)
    a[n // 2: 3 * n // 4] = (d[n // 2: 3 * n // 4] * np.exp2(rng.integers(-24, 4, n // 4))).astype(np.float32)
    e = edges()
    ea, ed = (g.ravel() for g in np.meshgrid(e, e))
    a, d = np.concatenate([a, ea, -ea]), np.concatenate([d, ed, ed])
    assert (np.abs(a) >= 2.0 ** -100).all()
    assert np.array_equal(bits(b.solve_op(DIV, a, d)), bits(a / d))


def test_division_of_zero_and_tiny_numerators(b):
    """Zeros give a zero (of positive sign).  Below 2^-100 the residual a - b q,
    at most 2^-23 of a, is rounded to a multiple of 2^-149 at worst to nothing,
    so the quotient keeps the error of the first one, 1.5 ulp, and its last
    rounding: 2 spacings of the result."""
    rng = np.random.default_rng(8)
    d = np.exp(rng.uniform(np.log(1e-18), np.log(1e18), 1 << 20)).astype(np.float32)
    z = b.solve_op(DIV, np.where(np.arange(d.size) % 2, np.float32(0), np.float32(-0.0)), d)
    assert (bits(z) == 0).all()
    a = np.exp2(rng.uniform(-148.0, -100.0, d.size)).astype(np.float32) * rng.choice(np.float32([-1, 1]), d.size)
    got, want = b.solve_op(DIV, a, d), a / d
    assert (np.abs(got.astype(np.float64) - want) <= 2.0 * np.abs(np.spacing(want)).astype(np.float64)).all()
