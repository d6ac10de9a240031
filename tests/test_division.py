"""The kernels' FP64 division (ice3_physics.hpp: by) against the IEEE quotient: on the CPU from reciprocals
as far off as the hardware's may be, on the GPU with the hardware's own.

A reciprocal within e0 = 4.7e-8 of 1/b is within e0^2 + 2^-53 = 2.4e-15 of it after the Newton step,
a quotient by it within 2.6e-15, and the correction adds the quotient's error but for 2.4e-15 of it (and
2^-53 of the residual): the sum that is rounded is within 7e-30 of a/b.  So the result is the IEEE quotient
unless a/b is that close to a rounding boundary, half an ulp from two neighbours, and then it is one of
them."""
import ctypes
import math
import os
import sys
from fractions import Fraction

import numpy as np
import pytest

sys.path.insert(0, os.path.join(os.path.dirname(os.path.abspath(__file__)), "host_stages"))
import host_lib  # noqa: E402

E0 = 4.7e-8
INF, NAN = np.inf, np.nan


def _pairs(n, seed):
    """Values over 2^+-300, and short mantissas (quotients that are exact or repeat)."""
    rng = np.random.Generator(np.random.Philox(seed))
    a, b = (np.ldexp(rng.uniform(1.0, 2.0, n) * rng.choice([-1.0, 1.0], n), rng.integers(-300, 301, n)) for _ in "ab")
    m = n // 4
    a[:m], b[:m] = rng.integers(-2 ** 20, 2 ** 20, m), rng.integers(1, 2 ** 20, m)
    a[m:2 * m] = np.nextafter(b[m:2 * m], np.where(rng.random(m) < 0.5, INF, -INF))  # quotients beside 1
    return a, b


def _hard_pairs(n, seed):
    """Pairs whose quotient is closest to the middle between two doubles: odd b and q with
    b (2 q + 1) = +-1 (mod 2^54), so that a = (b (2 q + 1) -+ 1) / 2^54 is a whole number."""
    rng = np.random.Generator(np.random.Philox(seed))
    out = []
    while len(out) < n:
        b = int(rng.integers(2 ** 52, 2 ** 53)) | 1
        for s in (1, -1):
            t = s * pow(b, -1, 2 ** 54) % 2 ** 54      # 2 q + 1, b t = s (mod 2^54)
            if t < 2 ** 53:
                continue
            a = (b * t - s) >> 54
            if 2 ** 52 <= a < 2 ** 53:
                out.append((float(a), float(b)))
    return tuple(np.array(v) for v in zip(*out[:n]))


def _neighbours(q, a, b):
    """Whether each q is one of the two doubles around a/b (or it), in exact arithmetic."""
    for x, y, z in zip(a.tolist(), b.tolist(), q.tolist()):
        e = Fraction(x) / Fraction(y)
        lo, hi = Fraction(math.nextafter(z, -INF)), Fraction(math.nextafter(z, INF))
        if not lo < e < hi:
            return False
    return True


def _host(a, b, r0):
    a, b, r0 = (np.ascontiguousarray(np.broadcast_to(v, np.shape(a)), dtype=np.float64) for v in (a, b, r0))
    q = np.empty_like(a)
    p = lambda v: ctypes.c_void_p(v.ctypes.data)  # noqa: E731
    f = host_lib.load().hst_quotients
    f.argtypes = [ctypes.c_void_p] * 4 + [ctypes.c_long]
    f(p(a), p(b), p(r0), p(q), a.size)
    return q


@pytest.mark.parametrize("off", [0.0, E0, -E0, "random"])
def test_quotients_from_any_reciprocal_within_the_bound(off):
    a, b = _pairs(1 << 20, 1)
    e = np.random.Generator(np.random.Philox(2)).uniform(-E0, E0, a.size) if off == "random" else off
    assert np.array_equal(_host(a, b, (1.0 / b) * (1.0 + e)), a / b)
    a, b = _hard_pairs(2000, 3)
    e = e[:a.size] if off == "random" else e
    assert _neighbours(_host(a, b, (1.0 / b) * (1.0 + e)), a, b)


def test_special_divisors():
    a = np.array([1.0, -1.0, 0.0, 2.5, 1.0, 1.0])
    b = np.array([0.0, -0.0, 0.0, INF, -INF, NAN])
    with np.errstate(divide="ignore"):
        assert np.isnan(_host(a, b, 1.0 / b)).all()
    assert np.array_equal(_host(np.zeros(3), [3.0, -7.0, 1e200], [1 / 3.0, -1 / 7.0, 1e-200]), np.zeros(3))


def test_no_values_is_a_call():
    from ice3_amd import _lib
    lib = _lib.load()
    assert lib.ice3_divide(0, None, None, None, None) == _lib.ICE3_OK
    assert lib.ice3_divide(-1, None, None, None, None) == _lib.ICE3_EINVAL
    assert lib.ice3_divide(1, None, None, None, None) == _lib.ICE3_EINVAL


@pytest.mark.gpu
def test_division_on_the_gpu():
    torch = pytest.importorskip("torch")
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from ice3_amd import _lib
    from ice3_amd._fields import ptr

    def run(a, b):
        x, y = (torch.from_numpy(np.ascontiguousarray(v, dtype=np.float64)).cuda() for v in (a, b))
        q = torch.full_like(x, -7.0)
        assert _lib.load().ice3_divide(x.numel(), ptr(x), ptr(y), ptr(q), None) == _lib.ICE3_OK
        torch.cuda.synchronize()
        return q.cpu().numpy()

    for seed in range(8):
        a, b = _pairs((1 << 21) + 77, 10 + seed)
        assert np.array_equal(run(a, b), a / b), seed
    a, b = _hard_pairs(4000, 20)
    q = run(a, b)
    assert _neighbours(q, a, b)
    print(f"division: {int((q != a / b).sum())} of {a.size} quotients at the middle of two doubles go the other way")
    assert np.isnan(run([1.0, -1.0, 0.0, 2.5, 1.0, 1.0], [0.0, -0.0, 0.0, INF, -INF, NAN])).all()
    assert np.array_equal(run([0.0, -0.0, 0.0], [3.0, -7.0, 1e200]), np.zeros(3))
