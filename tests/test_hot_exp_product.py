"""The exponential of a product without a table (csrc/staf_tri.hpp, HotExp<double>::product), which the fingerprints take for
exponents beyond the rows of their tables: re-evaluated here with exact fused multiply-adds and compared with exp(a y), the product taken
exactly."""
import math
import re
from decimal import Decimal

import numpy as np
import pytest

from test_hot_exp import SRC, fma


def source():
    s = open(SRC).read()
    body = s[s.index("__device__ static double eval(double x) {"):]
    body = body[:body.index("return ldexp")]
    co = [float(v) for v in re.findall(r"(?:scalar|vector)\(([0-9.eE+-]+)\)", body)]
    hi, lo = (float(v) for v in re.findall(r"fma\(t, -([0-9.eE+-]+), [xr]\)", body))
    product = s[s.index("__device__ static double product(double a, double y) {"):]
    top = float(re.search(r"e <= ([0-9.e+]+) \? fma\(e, fma\(a, y, -x\), e\) : e;", product).group(1))
    return co, hi, lo, top


def evaluate(a, y):
    co, hi, lo, top = source()
    x = a * y
    t = float(np.rint(x * 1.4426950408889634))
    r = fma(t, -lo, fma(t, -hi, x))
    p = co[0]
    for c in co[1:] + [0.5, 1.0, 1.0]:
        p = fma(p, r, c)
    try:
        e = math.ldexp(p, int(t))
    except OverflowError:   # (Python's ldexp; the instruction gives infinity)
        e = math.inf
    return fma(e, fma(a, y, -x), e) if e <= top else e


@pytest.mark.parametrize("size", [1e-3, 2.0, 17.0, 60.0, 600.0])
def test_against_exp_of_the_exact_product(size):
    """eval itself is off by 2e-16 at most (test_hot_exp); the last step rounds once more, 2^-53.  The rounding of a y that is made good
    would be up to 600 * 2^-53; its square is 5e-27."""
    rng = np.random.Generator(np.random.Philox(12))
    for a, y in zip(rng.uniform(-size, size, 400), rng.uniform(0, 1, 400)):
        want = (Decimal(float(a)) * Decimal(float(y))).exp()
        err = abs((Decimal(evaluate(float(a), float(y))) - want) / want)
        assert err <= Decimal(2e-16 + 2.0 ** -53), (a, y, err)


def test_limits():
    assert evaluate(0.0, 1.0) == 1.0 and evaluate(-800.0, 0.99) < 1e-300
    assert evaluate(1500.0, 0.7) == math.inf and evaluate(710.0, 1.0) == math.inf
