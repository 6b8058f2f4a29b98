"""The kernels' division by the lattice constants (fast_div) equals the IEEE
quotient, and the FP32 equilibria with it those with IEEE division, bit for
bit (tests/constdiv_check.c); in FP64 by a proof over the significands."""
import math
import os
import random
import shutil
import subprocess
from fractions import Fraction

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.mark.skipif(shutil.which("gcc") is None, reason="needs gcc")
def test_constant_division_is_exact(tmp_path):
    exe = str(tmp_path / "constdiv_check")
    subprocess.run(["gcc", "-O2", "-ffp-contract=off", "-mfma", os.path.join(HERE, "constdiv_check.c"), "-o", exe,
                    "-lm"], check=True)
    out = subprocess.run([exe, "2000000"], check=True, capture_output=True, text=True)
    rows = [line.split() for line in out.stdout.strip().splitlines()]
    assert len(rows) == 9
    for name, tested, bad in rows:
        assert int(tested) > 1_000_000 and int(bad) == 0, (name, tested, bad)


def _double_candidates(y, low):
    """Every significand X in [2^52, 2^53) whose quotient by the double y comes
    so close to the middle M of two doubles that x r + RN(x l) may round to the
    other side. |RN(x l) - x (1/y - r)| <= 2^-52 |x l|, so those have |rho| <= R
    = 2^55 |l y| in X 2^j - M Y = rho (Y y's significand, M odd in (2^53, 2^54),
    j = 53 or 54 as X >= Y or not): M is fixed modulo 2^j by each rho."""
    Y = int(math.frexp(y)[0] * 2**53)
    t = (Y & -Y).bit_length() - 1
    R = math.ceil(abs(Fraction(low) * Fraction(y)) * 2**55) + 1
    for j in (53, 54):
        mod = 1 << (j - t)
        inv = pow(Y >> t, -1, mod)
        for rho in range(-R, R + 1):
            if rho % (1 << t):
                continue
            m0 = (-(rho >> t) * inv) % mod
            for M in range(m0 + (2**53 - m0 + mod - 1) // mod * mod, 2**54, mod):
                X, left = divmod(rho + M * Y, 1 << j)
                if M % 2 and left == 0 and 2**52 <= X < 2**53 and (X >= Y) == (j == 53):
                    yield X


@pytest.mark.parametrize("lattice", ["d2q9", "d2q13"])
def test_double_constant_division_is_exact(lattice):
    """The same method in FP64: of all 2^52 significands only those near a
    rounding boundary can fail, and each of these is tried in exact
    arithmetic (float of a Fraction rounds to nearest even)."""
    C = 1.0 / math.sqrt(2.0 if lattice == "d2q13" else 3.0)
    c2 = C * C
    c4 = c2 * c2
    for y in (c2, 2 * c4, 2 * c2, 2 * (c2 * c4)):
        r = 1.0 / y
        low = float((1 - Fraction(r) * Fraction(y)) / Fraction(y))
        for X in _double_candidates(y, low):
            q = float(Fraction(X) * Fraction(r) + Fraction(float(X) * low))
            assert q == float(X) / y, (lattice, y, X)
        rng = random.Random(1)
        for _ in range(2000):
            X = rng.randrange(2**52, 2**53)
            assert float(Fraction(X) * Fraction(r) + Fraction(float(X) * low)) == float(X) / y
