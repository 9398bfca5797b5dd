"""The device forms of scream_amd/csrc/p3_math.h against the CPU's bits: the elementary
functions over and beyond P3's arguments and at special values, and the divisions in the
ranges they are stated for."""
import ctypes as C
import os

import numpy as np
import pytest

import oracle

pytestmark = pytest.mark.gpu

SUB, NORMAL, BIG = 5e-324, 2.2250738585072014e-308, 1.7976931348623157e308
SPECIAL = [0.0, -0.0, SUB, -SUB, 3e-310, NORMAL, -NORMAL, 1.0, -1.0, 1.0 - 2.0 ** -53, 1.0 + 2.0 ** -52, 2.0, -2.0, 0.5,
           1.4142135623730951, 0.7071067811865476, 4.0, 3.0, 1e300, -1e300, BIG, -BIG, np.inf, -np.inf, np.nan,
           709.782712893384, 709.7827128933841, -745.1332191019411, -745.1332191019412, -745.1332191019413, -708.4, 171.6,
           171.61, 170.0, 22.0, 22.1, -40.0, -40.1, 3.7e-9, 3.8e-9, 2.0 ** 31, 2.0 ** 53 + 2, 1e17]
EXP, LOG, LOG10, POW, CBRT, TGAMMA, EXPM1, TANH, DIV, DIV_INF, DIV_ANY, DIV_N, LOG10_POS, POW_LOG = range(14)


@pytest.fixture(scope="module")
def lib():
    import torch
    assert torch.cuda.is_available()
    d = C.CDLL(os.path.join(os.path.dirname(oracle.__file__), "libp3mathdev.so"))
    ptr = np.ctypeslib.ndpointer(np.float64, flags="C_CONTIGUOUS")
    d.p3md_eval.argtypes = [C.c_int, C.c_int, ptr, ptr, ptr]
    d.p3md_host.argtypes = [C.c_int, C.c_double, C.c_double]
    d.p3md_host.restype = C.c_double
    return d


def _device(lib, fn, x, y):
    x, y = (np.ascontiguousarray(a, np.float64) for a in np.broadcast_arrays(x, y))
    out = np.empty_like(x)
    assert lib.p3md_eval(fn, x.size, x, y, out) == 0
    return x, y, out


def _same(got, want, x, y, what):
    bad = np.flatnonzero((got.view(np.int64) != want.view(np.int64)) & ~(np.isnan(got) & np.isnan(want)))
    assert bad.size == 0, f"{what}: {bad.size} differ, e.g. " + ", ".join(
        f"({x[i]!r}, {y[i]!r}) device {got[i]!r} CPU {want[i]!r}" for i in bad[:4])


def _log_uniform(rng, lo, hi, n):
    return 10.0 ** rng.uniform(lo, hi, n)


ARGS = [
    (EXP, lambda r, n: (np.concatenate([r.uniform(-760, 720, n), _log_uniform(r, -320, 308, n) * r.choice([-1, 1], n)]), 0.0)),
    (LOG, lambda r, n: (np.concatenate([_log_uniform(r, -323, 308, n), r.uniform(0.5, 2, n), r.uniform(150, 350, n)]), 0.0)),
    (LOG10, lambda r, n: (np.concatenate([_log_uniform(r, -323, 308, n), _log_uniform(r, -25, 25, n)]), 0.0)),
    (POW, lambda r, n: (np.concatenate([_log_uniform(r, -300, 300, n), _log_uniform(r, -8, 8, n), -_log_uniform(r, -3, 3, n)]),
                        np.concatenate([r.uniform(-3, 3, n), r.uniform(-60, 60, n), r.integers(-20, 20, n) + 0.0]))),
    (CBRT, lambda r, n: (_log_uniform(r, -270, 308, n) * r.choice([-1, 1], n), 0.0)),
    (TGAMMA, lambda r, n: (np.concatenate([r.uniform(0, 30, n), r.uniform(30, 172, n), -r.uniform(0, 5, n)]), 0.0)),
    (EXPM1, lambda r, n: (np.concatenate([r.uniform(-1, 1, n), r.uniform(-50, 720, n), _log_uniform(r, -300, 0, n)]), 0.0)),
    (TANH, lambda r, n: (np.concatenate([r.uniform(-25, 25, n), _log_uniform(r, -12, 0, n) * r.choice([-1, 1], n)]), 0.0)),
    (LOG10_POS, lambda r, n: (_log_uniform(r, -323, 308, n), 0.0)),
    (POW_LOG, lambda r, n: (r.uniform(150, 350, n), r.uniform(-200, 200, n))),
]


@pytest.mark.parametrize("fn,args", ARGS, ids=[a[0] for a in ARGS])
def test_function_bits(lib, fn, args):
    x, y = args(np.random.default_rng(50 + fn), 20000)
    if fn not in (LOG10_POS, POW_LOG):
        x = np.concatenate([x, SPECIAL])
        if fn == POW:
            y = np.concatenate([y, np.resize([0.0, 1.0, 2.0, -0.5], len(SPECIAL))])
            xs, ys = (a.ravel() for a in np.meshgrid(SPECIAL, SPECIAL))
            x, y = np.concatenate([x, xs]), np.concatenate([y, ys])
    x, y, got = _device(lib, fn, x, y)
    cpu = oracle.load_oracle("portable").p3o_elementary if fn <= TANH else lib.p3md_host
    want = np.array([cpu(fn, float(a), float(b)) for a, b in zip(x, y)])
    _same(got, want, x, y, f"function {fn}")


def _operands(rng, n, lo, hi):
    """Operands with exponents from lo to hi, random significands and signs, and the specials."""
    def one():
        v = np.ldexp(rng.uniform(1, 2, n), rng.integers(lo, hi, n)) * rng.choice([-1.0, 1.0], n)
        return np.where(rng.random(n) < 0.02, rng.choice(SPECIAL, n), v)
    return one(), one()


def _divide(a, b):
    with np.errstate(all="ignore"):
        return a / b


def test_division_any(lib):
    rng = np.random.default_rng(1)
    for lo, hi in ((-1074, 1024), (-60, 60), (-1074, -1000)):
        a, b = _operands(rng, 200000, lo, hi)
        a, b, got = _device(lib, DIV_ANY, a, b)
        _same(got, _divide(a, b), a, b, f"any 2^{lo}..2^{hi}")


@pytest.mark.parametrize("fn", [DIV, DIV_INF])
def test_division_in_range(lib, fn):
    rng = np.random.default_rng(2)
    for lo, hi in ((-500, 500), (-1022, 1022), (-60, 60)):
        a, b = _operands(rng, 200000, lo, hi)
        q = _divide(a, b)
        plain = np.isfinite(a) & np.isfinite(b) & (a != 0) & (b != 0)
        normal = (np.abs(q) >= NORMAL) & np.isfinite(q) & (np.abs(b) >= NORMAL) & (np.abs(b) <= 2.0 ** 1022)
        keep = ~plain | (normal & (np.abs(a) >= 2.0 ** -969))  # zero, infinite and NaN operands too
        a, b = a[keep], b[keep]
        a, b, got = _device(lib, fn, a, b)
        _same(got, _divide(a, b), a, b, f"division {fn} 2^{lo}..2^{hi}")


def test_division_inf_outside(lib):
    """An overflowing quotient is infinite, also from a subnormal divisor, and a small
    dividend costs at most one unit in the last place."""
    rng = np.random.default_rng(3)
    a, b = _operands(rng, 200000, -1074, 1024)
    q = _divide(a, b)
    keep = np.isinf(q) & np.isfinite(a) & (b != 0)
    x, y, got = _device(lib, DIV_INF, a[keep], b[keep])
    _same(got, q[keep], x, y, "overflow")
    a = np.ldexp(rng.uniform(1, 2, 200000), rng.integers(-1074, -969, 200000))
    b = np.ldexp(rng.uniform(1, 2, 200000), rng.integers(-900, 0, 200000))
    for fn in (DIV, DIV_INF):
        a, b, got = _device(lib, fn, a, b)
        assert (np.abs(got - a / b) <= np.spacing(np.abs(a / b))).all()
