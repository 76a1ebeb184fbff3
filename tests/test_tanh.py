"""The hyperbolic tangent of the network kernel (csrc/staf_mlp_dev.hip, m_tanh in both precisions), re-evaluated on the CPU
from the constants in the source with correctly rounded fused multiply-adds: Cody-Waite reduction of 2|x| by ln 2, e^r - 1
by its Taylor polynomial, Newton-Raphson quotient.  The hardware reciprocal that the quotient starts from is taken off by
as much as its documentation allows, both ways.  The kernel itself is compared with the host evaluation on the GPU."""
import math
import os
import re
from decimal import Decimal, getcontext
from fractions import Fraction

import numpy as np
import pytest

SRC = os.path.join(os.path.dirname(__file__), "..", "alphanesgpu_amd", "csrc", "staf_mlp_dev.hip")
getcontext().prec = 50


def source(name):
    s = open(SRC).read()
    body = s[s.index(f"__device__ inline {name} m_tanh({name} x)"):]
    body = body[:body.index("return copysign")]
    num = lambda v: [float(a) / float(b or 1) for a, b in re.findall(r"([0-9.eE+-]+)f?(?: / ([0-9.]+)f?)?", v)][0]
    hi, lo = (num(v) for v in re.findall(r"fmaf?\(n, -([0-9.e+-]+)f?, [yr]\)", body))
    poly = [re.search(r"p = (1\.0f? / [0-9.]+)f?;", body).group(1)] + re.findall(r"p = fmaf?\(p, r, ([0-9.f/ ]+)\);", body)
    return dict(hi=hi, lo=lo, inv=num(re.search(r"rintf?\(y \* ([0-9.]+)f?\)", body).group(1)), poly=[num(v) for v in poly],
                top=num(re.search(r"> ([0-9.]+)f? \?", body).group(1)), newton=len(re.findall(r"q = fmaf?\(fmaf?\(-d, q", body)))


@pytest.mark.parametrize("name,rnd,eps,rcp,bound", [("double", np.float64, 2.0 ** -52, 2.0 ** -14, 1.6),
                                                    ("float", np.float32, 2.0 ** -23, 2.0 ** -22, 1.4)])
def test_reevaluated_tanh(name, rnd, eps, rcp, bound):
    c = source(name)
    R = lambda v: float(rnd(v))
    fma = lambda a, b, d: R(float(Fraction(a) * Fraction(b) + Fraction(d)))
    for k, v in enumerate(c["poly"]):      # the Taylor coefficients down to 1/2!
        assert R(v) == R(1.0 / math.factorial(len(c["poly"]) + 1 - k))
    rng = np.random.Generator(np.random.Philox(8))
    xs = np.concatenate([rng.uniform(-1, 1, 1500), rng.uniform(-12, 12, 800), 10.0 ** rng.uniform(-30, 0, 700),
                         [c["top"] / 2, 30.0, 1e30, 0.0]])
    worst = 0.0
    for x in (R(v) for v in xs):
        y = min(R(2 * abs(x)), c["top"])
        n = float(np.rint(R(y * R(c["inv"]))))
        r = fma(n, -R(c["lo"]), fma(n, -R(c["hi"]), y))
        p = R(c["poly"][0])
        for v in c["poly"][1:]:
            p = fma(p, r, R(v))
        p = fma(p, R(r * r), r)
        s = math.ldexp(1.0, int(n))
        m = fma(s, p, R(s - 1.0))
        d = R(m + 2.0)
        e = (Decimal(2 * abs(x)).exp() if abs(x) < 100 else Decimal(10) ** 60)
        # (below 1e-10 the difference of the exponentials cancels: x - x^3/3)
        want = Decimal(abs(x)) - Decimal(abs(x)) ** 3 / 3 if abs(x) < 1e-10 else (e - 1) / (e + 1)
        for off in (-rcp, rcp):
            q = R((1.0 + off) / d)
            for _ in range(c["newton"]):
                q = fma(fma(-d, q, 1.0), q, q)
            t = R(m * q)
            t = fma(fma(-d, t, m), q, t)
            if x == 0:
                assert t == 0
                continue
            worst = max(worst, float(abs(Decimal(t) - want) / want) / eps)
    assert worst < bound, worst
