"""The order in which the pressure solve sums its three Adams-Bashforth terms
(acme-ecp_amd/csrc/crm_round.hpp), built for the host.  The order decides the last bit of the
velocities, so it is fixed for every shape, engine and component: the product that is rounded by
itself, then two fused multiply-adds.  Expected values: exact rational arithmetic, rounded where
the order rounds.  The operands are the scheme's coefficients with terms that nearly cancel, where
the orders give different bits."""
import os
import subprocess
from fractions import Fraction

import numpy as np

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def alone(columns, y3, fp64, field):
    """The term whose product is rounded by itself."""
    if columns == 64:
        return "c" if field != "v" else "a" if fp64 else "b"
    if columns == 128 or y3:
        return "b"
    return {"u": "b", "w": "a"}[field]


def expected(term, v):
    at, a, bt, b, ct, c = (Fraction(x) for x in v)

    def fma(x, y, z):
        return Fraction(float(x * y + z))

    if term == "a":
        return float(fma(ct, c, fma(bt, b, Fraction(float(at * a)))))
    if term == "b":
        return float(fma(ct, c, fma(at, a, Fraction(float(bt * b)))))
    return float(fma(at, a, fma(bt, b, Fraction(float(ct * c)))))


def test_adams_bashforth_sums(tmp_path):
    exe = tmp_path / "round_check"
    subprocess.run(["g++", "-O2", "-std=c++17", "-I", os.path.join(ROOT, "acme-ecp_amd", "csrc"),
                    "-o", str(exe), os.path.join(ROOT, "tests", "native", "round_check.cpp")], check=True)
    rng = np.random.default_rng(1)
    ct = 5.0 / 12.0
    bt = -(1.0 + 4.0 * ct) / 2.0
    at = 1.0 - bt - ct
    ops = []
    for a, b in rng.uniform(-1.0, 1.0, (20, 2)):
        ops.append([at, a, bt, b, ct, float(-(at * a + bt * b) / ct)])
    text = "\n".join(" ".join(float(x).hex() for x in v) for v in ops)
    out = subprocess.run([str(exe)], input=text, check=True, capture_output=True, text=True).stdout.split("\n")
    # columns x 3D x engine x component: 5 2D shapes of two components, 2 3D shapes of three
    per = 2 * (5 * 2 + 2 * 3)
    assert len(out) == per * len(ops) + 1
    told_apart = set()
    for j, v in enumerate(ops):
        told_apart |= {s + t for s, t in ("ab", "ac", "bc") if expected(s, v) != expected(t, v)}
        for line in out[j * per:(j + 1) * per]:
            columns, y3, fp64, field, bits = line.split()
            want = expected(alone(int(columns), y3 == "1", fp64 == "1", field), v)
            assert float.fromhex(bits) == want, line
    assert told_apart == {"ab", "ac", "bc"}  # by these operands
