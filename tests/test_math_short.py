"""The short evaluation of the device's log / exp / pow and its rounding test: what it accepts has the
double-double path's bits, and arguments that it rejects (one in 8,000 for exp and pow, 41,000 for log over
the path's ranges, found here by running it on the host) take that path, on the host and on the device."""
import ctypes as C

import numpy as np
import pytest

import oracle as O
from openradioss_amd import engine as E

FN = {"log": 0, "exp": 1, "pow": 2}


def _p(a):
    return None if a is None else a.ctypes.data_as(C.c_void_p)


def short(fn, x, y=None):
    """(value, accepted) of the short evaluation."""
    out, acc = np.empty_like(x), np.empty(x.size, np.uint8)
    O.lib("cr").or_short_eval(C.c_int(FN[fn]), C.c_int64(x.size), _p(x), _p(y), _p(out), _p(acc))
    return out, acc.astype(bool)


def evaluate(name, fn, x, y=None):
    out = np.empty_like(x)
    getattr(O.lib("cr"), name)(C.c_int(FN[fn]), C.c_int64(x.size), _p(x), _p(y), _p(out))
    return out


def arguments(fn, n, seed):
    """Arguments over the ranges the path uses."""
    rng = np.random.default_rng(seed)
    if fn == "log":
        return np.exp(rng.uniform(-40.0, 25.0, n)), None
    if fn == "exp":
        return rng.uniform(-60.0, 12.0, n), None
    y = np.where(rng.integers(0, 2, n) == 0, rng.choice([1.0 / 3.0, 2.0 / 3.0], n), rng.uniform(-1.0, 1.0, n))
    return np.exp(rng.uniform(-30.0, 14.0, n)), y


def rejected(fn, n=4_000_000):
    x, y = arguments(fn, n, 31 + FN[fn])
    no = ~short(fn, x, y)[1]
    return x[no], None if y is None else y[no]


@pytest.mark.parametrize("fn", list(FN))
def test_accepted_values_have_the_double_double_bits(fn):
    x, y = arguments(fn, 1_000_000, 7)
    out, acc = short(fn, x, y)
    assert 0.999 < acc.mean() < 1.0
    assert np.array_equal(out[acc], evaluate("or_cr_eval", fn, x, y)[acc])


@pytest.mark.parametrize("fn", list(FN))
def test_rejected_arguments_take_the_double_double_path(fn):
    x, y = rejected(fn)
    assert x.size >= 50
    assert np.array_equal(evaluate("or_device_eval", fn, x, y), evaluate("or_cr_eval", fn, x, y))


def test_two_powers_of_which_one_is_rejected():
    x, y = arguments("pow", 4_000_000, 5)
    n = np.random.default_rng(6).uniform(0.0, 1.0, x.size)
    check = O.lib("cr").or_device_pow2_check
    check.restype = C.c_int64
    for y1, y2 in ((n, 1.0 - n), (np.full_like(n, 1.0 / 3.0), np.full_like(n, 2.0 / 3.0))):
        a, b = short("pow", x, y1)[1], short("pow", x, y2)[1]
        for some in (a & ~b, ~a & b):
            assert some.sum() >= 100
            v, w1, w2 = x[some], y1[some], y2[some]
            assert check(C.c_int64(v.size), _p(v), _p(w1), _p(w2)) == 0


@pytest.mark.gpu
@pytest.mark.parametrize("fn", list(FN))
def test_rejected_arguments_on_the_device(fn, gpu_lib):
    x, y = rejected(fn)
    print(f"case: or_math_eval {fn}, {x.size} arguments that the rounding test rejects", flush=True)
    assert x.size >= 50
    assert np.array_equal(E.math_eval(fn, x, y), evaluate("or_cr_eval", fn, x, y))
