"""The exponential of a product whose factor is held in two parts (csrc/staf_tri.hpp, HotExp<double>::Factor): its
constants are read from the source, the function is re-evaluated here with exact fused multiply-adds and compared with
exp(a y), the product taken exactly.  The kernels themselves are compared with the oracle on the GPU."""
import math
import os
import re
from decimal import Decimal

import numpy as np
import pytest

from test_hot_exp import SRC, fma, source_constants


def factor_constants():
    s = open(SRC).read()
    s = s[s.index("struct Factor { double hi, lo; };"):]
    unit = float(re.search(r"const double hi = a \* ([0-9.eE+-]+);", s).group(1))
    low = float(re.search(r"fma\(a, ([0-9.eE+-]+), fma\(a, " + re.escape(repr(unit)) + r", -hi\)\)", s).group(1))
    body = s[s.index("double q = "):s.index("return ldexp(fma(g, q * r, g)")]
    co = [float(v) for v in re.findall(r"\b[0-9]\.[0-9]+(?:e-[0-9]+)?", body)]
    assert len(co) == 5 and co[1] == co[2]   # (one of them stands in both branches of a choice)
    return unit, low, [co[0], co[1], co[3], co[4]]


def evaluate(a, y):
    table = source_constants()[0]
    unit, low, co = factor_constants()
    hi = a * unit
    lo = fma(a, low, fma(a, unit, -hi))
    t = float(np.rint(y * hi))
    r = fma(y, lo, fma(y, hi, -t))
    i = int(t)
    q = co[0]
    for c in co[1:]:
        q = fma(q, r, c)
    return math.ldexp(fma(table[i & 127], q * r, table[i & 127]), i >> 7)


def test_the_unit_is_128_over_ln2_in_two_parts():
    unit, low, _ = factor_constants()
    want = 128 / Decimal(2).ln()
    assert unit == float(want) and low == float(want - Decimal(unit))


@pytest.mark.parametrize("size", [1e-3, 0.05, 2.0, 60.0, 600.0])
def test_against_exp_of_the_exact_product(size):
    """Roundings of the table value and of the last step, half a unit in the last place each (2^-53), and the truncation,
    7.6e-17; what the rounding of q adds is below 2^-53 * 0.003."""
    rng = np.random.Generator(np.random.Philox(11))
    a = rng.uniform(-size, size, 800)
    y = np.concatenate([rng.uniform(0, 1, 790), [0.0, 1.0, 1e-300, 1e-17, 0.5, 2.0 ** -30, 0.999, 1e-5, 0.25, 0.75]])
    for a_, y_ in zip(a, y):
        want = (Decimal(float(a_)) * Decimal(float(y_))).exp()
        err = abs((Decimal(evaluate(float(a_), float(y_))) - want) / want)
        assert err <= Decimal(2 * 2.0 ** -53 + 7.6e-17 + 4e-19), (a_, y_, err)


def test_limits():
    assert evaluate(0.0, 1.0) == 1.0 and evaluate(3.0, 0.0) == 1.0 and evaluate(-0.0, 0.0) == 1.0
    assert evaluate(-1000.0, 1.0) == 0.0
    with pytest.raises(OverflowError):   # (Python's ldexp; the instruction gives infinity)
        evaluate(1000.0, 1.0)
