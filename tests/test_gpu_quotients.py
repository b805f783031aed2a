"""The kernels' shared-denominator quotients and square root against numpy's
a / b and sqrt, bit for bit: mantissas and exponents at random over the stated
ranges, mantissas at their ends, and zeros, infinities and NaN."""
import ctypes as C
import os

import numpy as np
import pytest

from csu_amd import build

pytestmark = pytest.mark.gpu

SO = os.path.join(build.LIB, "libcsu_quotients.so")
N = 1 << 20


def _eval(op, a, b, rb):
    if not os.path.exists(SO):
        build.build_test_lib(os.path.join(os.path.dirname(os.path.abspath(__file__)), "quotients.hip"),
                             os.path.basename(SO))
    L = C.CDLL(SO)
    t = C.c_double if a.dtype == np.float64 else C.c_float
    f = L.quotients_f64 if a.dtype == np.float64 else L.quotients_f32
    arrs = [np.ascontiguousarray(x, a.dtype) for x in (a, b, rb)]
    out = np.empty_like(arrs[0])
    assert f(len(a), op, *[x.ctypes.data_as(C.POINTER(t)) for x in arrs], out.ctypes.data_as(C.POINTER(t))) == 0
    return out


def _same(x, y):
    u = np.uint64 if x.dtype == np.float64 else np.uint32
    return (np.isnan(x) & np.isnan(y)) | (x.view(u) == y.view(u))


def _random(rng, n, dtype, lo, hi):
    """Random signs and mantissas, an eighth of them within 4 ulp of a power
    of two, exponents lo .. hi - 1."""
    bits = 53 if dtype == np.float64 else 24
    m = rng.integers(1 << (bits - 1), 1 << bits, n)
    end = rng.random(n) < 0.125
    m[end] = np.where(rng.random(end.sum()) < 0.5, (1 << (bits - 1)) + rng.integers(0, 4, end.sum()),
                      (1 << bits) - 1 - rng.integers(0, 4, end.sum()))
    e = rng.integers(lo, hi, n)
    return (np.ldexp(m.astype(np.float64), e - bits + 1) * np.where(rng.random(n) < 0.5, -1.0, 1.0)).astype(dtype)


# numerators, denominators, quotients: powers of two of the stated ranges
RANGES = {np.float64: ((-960, 1000), (-1000, 1000), (-1000, 1000)),
          np.float32: ((-100, 120), (-120, 120), (-120, 120))}


@pytest.mark.parametrize("form", ["f64", "f64_given_reciprocal", "f32"])
def test_quotients(form):
    dtype = np.float32 if form == "f32" else np.float64
    ra, rb, rq = RANGES[dtype]
    rng = np.random.default_rng(11)
    a, b = _random(rng, N, dtype, *ra), _random(rng, N, dtype, *rb)
    near = rng.random(N) < 0.5           # exponents of half of them as close as the solver's
    b[near] = _random(rng, int(near.sum()), dtype, -30, 30)
    a[near] = _random(rng, int(near.sum()), dtype, -60, 60)
    special = np.array([0.0, -0.0, np.inf, -np.inf, np.nan, 1.0, -3.0], dtype)
    sa, sb = (x.ravel() for x in np.meshgrid(special, special))
    with np.errstate(all="ignore"):
        e = np.log2(np.abs(a.astype(np.float64))) - np.log2(np.abs(b.astype(np.float64)))
        keep = (e > rq[0]) & (e < rq[1])
        a, b = np.r_[a[keep], sa], np.r_[b[keep], sb]
        want = a / b
        out = _eval(1 if form.endswith("reciprocal") else 0, a, b, (1 / b).astype(dtype))
    bad = ~_same(out, want)
    assert keep.sum() > N // 4 and not bad.any(), (bad.sum(), a[bad][:3], b[bad][:3], out[bad][:3], want[bad][:3])


def test_square_root():
    rng = np.random.default_rng(12)
    a = np.abs(_random(rng, N, np.float64, -760, 1020))
    a[: N // 2] = np.abs(_random(rng, N // 2, np.float64, -40, 60))
    a = np.r_[a, [0.0, -0.0, np.inf, np.nan, -1.0, -np.inf, 1.0, 4.0]]
    with np.errstate(all="ignore"):
        want = np.sqrt(a)
    bad = ~_same(_eval(2, a, a, a), want)
    assert not bad.any(), (bad.sum(), a[bad][:3])
