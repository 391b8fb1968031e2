"""Static algorithmic FLOP count of the device RHS and of one Cash-Karp attempt.

The count is taken from the source text of the blocks of the RHS in
``galacticus_amd/csrc/physics.hpp`` (plus the sum that joins its two halves
and the inlined helpers), so it moves with the code.  Each block counts once,
whichever wave of a group computes it.  Weights:

* ``+ - * /`` on doubles, ``sqrt``, ``rsqrt``, ``fmin``, ``fmax``, ``fabs``: 1
* ``exp``, ``log``, ``log1p``, ``cbrt``, ``atan``, ``pow``, ``sinh``: 20 each
  (a fixed weight for a transcendental; the device implementations cost
  20-80 FP64 instructions)

Integer index arithmetic, comparisons and selects are not counted.  The RHS is
straight-line code, so every counted operation executes on every evaluation.

One Cash-Karp attempt on N=30 variables costs
``FLOP_step = 6*F_rhs + F_comb`` with ``F_comb = 52*N``: stage inputs
(1+2+3+4+5 products and sums per variable, times 2) plus the 5th-order
solution (4 terms) and the error (5 terms), times 2, plus 4 operations per
variable for the error norm.
"""
from __future__ import annotations

import os
import re

HERE = os.path.dirname(os.path.abspath(__file__))
PHYSICS = os.path.join(HERE, "csrc", "physics.hpp")
NVAR = 30
TRANSCENDENTAL_WEIGHT = 20
TRANSCENDENTALS = ("exp", "log", "log1p", "cbrt", "atan", "pow", "sinh")
UNIT_CALLS = ("sqrt", "rsqrt", "fmin", "fmax", "fabs")
# The functions an evaluation goes through once.
BLOCKS = ("halo", "time_part", "cooling_temperature_index", "cooling_cell", "cooling_function", "isco", "galaxy_radius",
          "hot_profile", "hot_inv_mean_radius", "black_hole", "cooling_time", "galaxy_rates", "outer_radius_rates",
          "hot_accretion", "accretion_rate", "jet_power", "black_hole_growth", "spheroid_shares", "spheroid_rates",
          "radiated_energy", "cooling_rates")


def _function_body(src: str, signature_start: str) -> str:
    i = src.index(signature_start)
    j = src.index("{", i)
    depth = 0
    for k in range(j, len(src)):
        if src[k] == "{":
            depth += 1
        elif src[k] == "}":
            depth -= 1
            if depth == 0:
                return src[j:k + 1]
    raise ValueError("unbalanced braces")


def _strip(body: str) -> str:
    body = re.sub(r"//[^\n]*", "", body)
    body = re.sub(r"#pragma[^\n]*", "", body)
    return body


def _count_ops(body: str) -> int:
    b = _strip(body)
    b = re.sub(r"\bfma\(", "fma(+*", b)              # a product and a sum
    b = re.sub(r"\[[^\]]*\]", "", b)                 # array indices are not flops
    b = re.sub(r"\+\+|--", "", b)
    b = re.sub(r"<=|>=|==|!=|&&|\|\||->", " ", b)
    arith = len(re.findall(r"(?<![eE])[+\-*/](?!=)", b)) + len(re.findall(r"[+\-*/]=", b))
    trans = sum(len(re.findall(r"\b%s\(" % f, b)) for f in TRANSCENDENTALS)
    unit = sum(len(re.findall(r"\b%s\(" % f, b)) for f in UNIT_CALLS)
    return arith + unit + TRANSCENDENTAL_WEIGHT * trans


def rhs_flops() -> int:
    src = open(PHYSICS, encoding="utf-8").read()
    def ops(name: str) -> int:
        return _count_ops(_function_body(src, re.search(
            r"__device__ __forceinline__ \w+ %s\(" % name, src).group(0)))

    total = sum(ops(name) for name in BLOCKS)
    total += 2 * ops("hernquist_density")   # at the accretion radius and at the Jeans length
    total += NVAR    # f = f_galaxy + f_halo
    total += 4 * 3   # pow_half: three multiplies (and one divide) per power law
    return total


def combination_flops(nvar: int = NVAR) -> int:
    return 52 * nvar


def attempt_flops() -> int:
    return 6 * rhs_flops() + combination_flops()


def evaluated_flops(rhs_evaluations: int, attempts: int) -> int:
    """Algorithmic FLOPs of a launch from its measured counters: every RHS
    evaluation (six for an accepted attempt, five for a rejected one, whose
    end-point derivative is never taken, plus the first of each node) and the
    stage combinations and error norm of every attempt."""
    return int(rhs_evaluations) * rhs_flops() + int(attempts) * combination_flops()


if __name__ == "__main__":
    print("F_rhs", rhs_flops(), "F_comb", combination_flops(), "FLOP_step", attempt_flops())
