"""Write hamx_sync_fine.h: the synchrotron kernels' series of
gen_hamx_synchrotron.py (P(u) = ln F + x and R(u) = G / F in u = ln x) on short
segments, as the march evaluates them: 72 segments of width 1/4 below
u = ln 100, each a degree-7 polynomial in v in [-1, 1] (Chebyshev
interpolation of the same extended-precision sums, converted to powers), P and
R interleaved.  Interpolation error below 4e-15 (a degree-6 series: 1e-13).

Run: python gen_hamx_sync_fine.py [output.h]   (numpy only; a few seconds)
"""
import sys

import numpy as np
from numpy.polynomial import chebyshev as cheb

from gen_hamx_synchrotron import U_TOP, target_p, target_r

N, WIDTH, DEGREE = 72, 0.25, 7


def powers(target, lo):
    nodes = np.cos(np.pi * (np.arange(DEGREE + 1) + 0.5) / (DEGREE + 1))
    vals = [target(lo + 0.5 * WIDTH * (1 + t)) for t in nodes]
    return cheb.cheb2poly(cheb.chebfit(nodes, np.array(vals), DEGREE))


def render() -> str:
    lines = [
        "// Generated by gen_hamx_sync_fine.py; do not edit.",
        "// P(u) = ln F(x) + x and R(u) = G(x) / F(x), u = ln x: segment s covers",
        "// [kUTop - (s + 1) w, kUTop - s w], w = kFineSegW; {P, R} coefficients of v^k,",
        "// v in [-1, 1] across the segment.",
        "#pragma once",
        "",
        "namespace hamx {",
        "namespace sync_tab {",
        f"constexpr int kFineSeg = {N};",
        f"constexpr double kFineSegW = {WIDTH!r};",
        f"constexpr int kFineSegDeg = {DEGREE};",
        "__device__ __constant__ const double kFineTab[kFineSeg][kFineSegDeg + 1][2] = {",
    ]
    for s in range(N):
        lo = U_TOP - (s + 1) * WIDTH
        cp, cr = powers(target_p, lo), powers(target_r, lo)
        lines.append("    {" + ", ".join(f"{{{float(a)!r}, {float(b)!r}}}"
                                         for a, b in zip(cp, cr)) + "},")
    lines += ["};", "} // namespace sync_tab", "} // namespace hamx", ""]
    return "\n".join(lines)


if __name__ == "__main__":
    out = sys.argv[1] if len(sys.argv) > 1 else __file__.replace(
        "gen_hamx_sync_fine.py", "hamx_sync_fine.h")
    with open(out, "w") as f:
        f.write(render())
    print("wrote", out)
