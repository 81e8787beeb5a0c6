"""The FP64 line sums take the Taylor polynomial of exp of degree 6, 8 or 10 up to a largest argument each
(line_degree in slgpu_opacity.hip).  At every limit the remainder relative to the exponential, of either
sign of the argument, is under 2^-53, as stated there.  Computed with 40 digits."""
import os
import re
from decimal import Decimal, getcontext
from math import factorial

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_remainders_at_the_limits():
    getcontext().prec = 40
    src = open(os.path.join(ROOT, "superlite_amd", "csrc", "slgpu_opacity.hip")).read()
    body = src[src.index("int line_degree("):]
    limits = re.findall(r"x <= ([0-9.]+) \? (\d+)", body[:body.index("\n}")])
    assert [int(n) for _, n in limits] == [6, 8, 10]
    for x, n in limits:
        for t in (Decimal(x), -Decimal(x)):
            p = sum(t ** k / factorial(k) for k in range(int(n) + 1))
            assert abs(p - t.exp()) / t.exp() < Decimal(2) ** -53, (x, n)
