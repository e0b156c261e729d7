"""Write hamx_sync_fine.h: the synchrotron kernels' series of
gen_hamx_synchrotron.py (P(u) = ln F + x and R(u) = G / F in u = ln x) on short
segments, as the march evaluates them: 72 segments of width 1/4 below
u = ln 100, each a degree-8 polynomial in v in [-1, 1] (Chebyshev
interpolation of the same sums and its powers, in extended precision throughout),
P and R interleaved.  Evaluated in 64 bits across the segments P is 1.3e-16 rms
off and 4.2e-16 at most, R 6.9e-17 and 2.2e-16 (relative); the Chebyshev series of
gen_hamx_synchrotron.py 3.3e-16 and 1.7e-15, 2.6e-16 and 1.2e-15.  Degree 7 is not
enough (5.9e-16 and 1.0e-15 rms), nor are interpolation and conversion in 64 bits
(1.0e-15 rms of P).

Run: python gen_hamx_sync_fine.py [output.h]   (numpy only; a few seconds)
"""
import sys

import numpy as np

from gen_hamx_synchrotron import U_TOP, ratio_r, sum_p

N, WIDTH, DEGREE = 72, 0.25, 8
LD = np.longdouble
PI = LD("3.14159265358979323846264338327950288")


def powers(target, lo):
    n = DEGREE + 1
    angle = PI * (np.arange(n).astype(LD) + LD(0.5)) / n
    vals = np.array([target(LD(lo) + LD(WIDTH) / 2 * (1 + t)) for t in np.cos(angle)])
    # T_k as powers, and the interpolant's coefficients by the discrete cosine sum
    cheb = [np.array([LD(1)]), np.array([LD(0), LD(1)])]
    for k in range(2, n):
        t = np.zeros(k + 1, dtype=LD)
        t[1:] = 2 * cheb[-1]
        t[:k - 1] -= cheb[-2]
        cheb.append(t)
    out = np.zeros(n, dtype=LD)
    for k in range(n):
        out[:k + 1] += (2 if k else 1) * np.sum(vals * np.cos(k * angle)) / n * cheb[k]
    return out


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
        cp, cr = powers(sum_p, lo), powers(ratio_r, lo)
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
