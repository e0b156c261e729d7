"""Write hamx_synchrotron.h: piecewise Chebyshev tables of the synchrotron
kernels F(x) = x * int_x^inf K_{5/3}(t) dt and G(x) = x K_{2/3}(x), the
functions the reference takes from GSL (gsl_sf_synchrotron_1 / _2,
integrator.cc:321,390).

F is fitted as P(u) = ln(F(x)) + x in u = ln x, so that F = exp(P - x) keeps
a uniform relative accuracy from the x^(1/3) rise at small x to the e^(-x)
tail at x = 100 (the largest argument the reference integrates,
integrator.cc:312-315); P varies slowly (dP/du stays below 1/2 + 1/3), so an
error in u moves F by less than that error.  G is fitted as the ratio
R(u) = G(x) / F(x), which stays between 1/2 (x -> 0) and 1, so G = F R
costs no second exponential.  Both use the same segments:

* u in [ln 100 - 9, ln 100]: 9 segments of width 1, degree 12;
* u in [ln 100 - 57, ln 100 - 9]: 12 segments of width 4, degree 16;
* below that (x < 1.8e-23) the leading terms F = 2^(2/3) Gamma(2/3) x^(1/3)
  and R = 1/2 (the next terms are O(x^(2/3)) relative, below 1e-15 there).

The fitted values come from the integral representations
  F(x) = x int_0^inf cosh(5s/3) / cosh(s) exp(-x cosh s) ds
  G(x) = x int_0^inf cosh(2s/3) exp(-x cosh s) ds
(int_x^inf K_nu = int_0^inf cosh(nu s)/cosh(s) e^{-x cosh s} ds follows from
K_nu(t) = int_0^inf e^{-t cosh s} cosh(nu s) ds), summed by the trapezoid rule
in extended precision: the integrands are analytic in a strip about the real
axis, so the rule converges exponentially (step 1/200, range [0, 80]).

Run: python gen_hamx_synchrotron.py [output.h]   (numpy only; a few seconds)
"""
import math
import sys

import numpy as np
from numpy.polynomial import chebyshev as cheb

U_TOP = math.log(100.0)
FINE = dict(n=9, width=1.0, degree=12)
COARSE = dict(n=12, width=4.0, degree=16)
H = np.longdouble(1) / 200
S = np.arange(0, 80, H, dtype=np.longdouble)
W_F = np.cosh(5 * S / 3) / np.cosh(S)
W_G = np.cosh(2 * S / 3)


def _trap(weight, x):
    f = weight * np.exp(-np.longdouble(x) * np.cosh(S))
    return np.longdouble(x) * H * (f.sum() - f[0] / 2)


def sum_p(u):
    x = np.exp(np.longdouble(u))
    return np.log(_trap(W_F, x)) + x


def ratio_r(u):
    x = np.exp(np.longdouble(u))
    return _trap(W_G, x) / _trap(W_F, x)


def target_p(u):
    return float(sum_p(u))


def target_r(u):
    return float(ratio_r(u))


def segments():
    """(lo, hi, degree) from the top of the range downwards."""
    out = []
    top = U_TOP
    for spec in (FINE, COARSE):
        for _ in range(spec["n"]):
            out.append((top - spec["width"], top, spec["degree"]))
            top -= spec["width"]
    return out


def fit(target):
    coefs = []
    for lo, hi, deg in segments():
        nodes = np.cos(np.pi * (np.arange(deg + 1) + 0.5) / (deg + 1))
        vals = [target(0.5 * (lo + hi) + 0.5 * (hi - lo) * t) for t in nodes]
        c = cheb.chebfit(nodes, np.array(vals), deg)
        coefs.append(list(c) + [0.0] * (COARSE["degree"] - deg))
    return coefs


def render() -> str:
    cf, cr = fit(target_p), fit(target_r)
    g23 = math.gamma(2.0 / 3.0)
    nseg = FINE["n"] + COARSE["n"]
    ncoef = COARSE["degree"] + 1
    lines = [
        "// Generated by gen_hamx_synchrotron.py; do not edit.",
        "// Piecewise Chebyshev tables in u = ln x of P(u) = ln F(x) + x and",
        "// R(u) = G(x) / F(x) for the synchrotron kernels F = x int_x^inf K_5/3",
        "// and G = x K_2/3.",
        "#pragma once",
        "",
        "namespace hamx {",
        "namespace sync_tab {",
        f"constexpr double kUTop = {U_TOP!r};",
        f"constexpr int kFineN = {FINE['n']};",
        f"constexpr double kFineW = {FINE['width']!r};",
        f"constexpr int kFineDeg = {FINE['degree']};",
        f"constexpr int kCoarseN = {COARSE['n']};",
        f"constexpr double kCoarseW = {COARSE['width']!r};",
        f"constexpr int kCoarseDeg = {COARSE['degree']};",
        f"constexpr int kSeg = {nseg};",
        f"constexpr int kCoef = {ncoef};",
        f"constexpr double kLnF0 = {math.log(2 ** (2 / 3) * g23)!r}; // ln(2^(2/3) Gamma(2/3))",
        "constexpr double kR0 = 0.5; // G / F as x -> 0",
    ]
    for name, tab in (("kF", cf), ("kR", cr)):
        lines.append(f"__device__ __constant__ const double {name}[kSeg][kCoef] = {{")
        for row in tab:
            lines.append("    {" + ", ".join(repr(float(v)) for v in row) + "},")
        lines.append("};")
    lines += ["} // namespace sync_tab", "} // namespace hamx", ""]
    return "\n".join(lines)


if __name__ == "__main__":
    out = sys.argv[1] if len(sys.argv) > 1 else __file__.replace(
        "gen_hamx_synchrotron.py", "hamx_synchrotron.h")
    with open(out, "w") as f:
        f.write(render())
    print("wrote", out)
