"""The polynomials of the logarithmic means without logarithms (csrc/physics.hpp,
log_free_means): the stored coefficients, read from the source, evaluated exactly
against 2 atanh(z)/z and its reciprocal up to the |z| = 0.15 they are used for."""
import os
import re
from fractions import Fraction

HERE = os.path.dirname(os.path.abspath(__file__))
SOURCE = os.path.join(os.path.dirname(HERE), "trixicuda.jl_amd", "csrc", "physics.hpp")


def _coefficients(variable, code):
    """Highest first: those of a Horner scheme in `variable`."""
    body = code[code.index(f"double {variable} = fma("):]
    lines = []
    for line in body.splitlines():
        if not re.match(rf"\s*(double )?{variable} = fma\(", line):
            break
        lines.append(line)
    numbers = re.findall(r"-?\d+\.\d+(?:e-?\d+)?", "\n".join(lines))
    return [Fraction(float(x)) for x in numbers]


def test_stored_polynomials():
    with open(SOURCE) as f:
        code = f.read()
    code = code[code.index("void log_free_means("):]
    Q, P = _coefficients("Q", code), _coefficients("Pq", code)
    assert len(Q) == len(P) == 7 and Q[-1] == Fraction(1, 2) and P[-1] == 2
    worst_p = worst_q = 0
    for i in range(1, 301):
        q = Fraction(15 * i, 30000) ** 2  # z^2, |z| up to 0.15
        exact = sum(2 * q**k / (2 * k + 1) for k in range(40))  # the rest is below 1e-65
        p_val = q_val = Fraction(0)
        for c in P:
            p_val = p_val * q + c
        for c in Q:
            q_val = q_val * q + c
        worst_p = max(worst_p, abs(p_val / exact - 1))
        worst_q = max(worst_q, abs(q_val * exact - 1))
    print(float(worst_p), float(worst_q))
    # as stated beside them: below half a unit in the last place
    assert worst_p < Fraction(52, 10**18) and worst_q < Fraction(11, 10**18)
