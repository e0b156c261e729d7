"""CPU check of the synchrotron kernels' short segments (hamx_sync_fine.h): the
polynomials as the device evaluates them (one rounding per fused step) against
the integral representations of F and G summed in extended precision.  They are
no further off than the Chebyshev series they replaced, which measured 3.3e-16
rms and 1.7e-15 at most in ln F + x, 2.6e-16 and 1.2e-15 in G / F: the bounds are
half of those, above half an ulp of the values (2.2e-16 up to 2.5) plus the last
product's rounding."""
import os
import re
import sys

import numpy as np

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                    "hammurabix_amd", "csrc")


def test_short_segments():
    sys.path.insert(0, CSRC)
    try:
        import gen_hamx_synchrotron as gen
    finally:
        sys.path.remove(CSRC)
    src = open(os.path.join(CSRC, "hamx_sync_fine.h")).read()
    n = int(re.search(r"kFineSeg = (\d+)", src).group(1))
    width = float(re.search(r"kFineSegW = ([\d.]+)", src).group(1))
    deg = int(re.search(r"kFineSegDeg = (\d+)", src).group(1))
    body = src[src.index("kFineTab["):]
    tab = np.array(re.findall(r"-?\d+\.\d+(?:e[-+]\d+)?", body), dtype=float)
    tab = tab.reshape(n, deg + 1, 2)
    # points across every segment, the ends among them
    u = gen.U_TOP - (np.repeat(np.arange(n), 6) +
                     np.tile([1e-9, 0.13, 0.37, 0.5, 0.81, 1 - 1e-9], n)) * width
    d = (gen.U_TOP - u) * (1 / width)
    s = d.astype(int)
    v = 2.0 * (s - d) + 1.0
    ld = np.longdouble
    want = np.array([(gen.sum_p(x), gen.ratio_r(x)) for x in u])
    for m, name, rms, worst in ((0, "ln F + x", 1.6e-16, 8.5e-16), (1, "G / F", 1.3e-16, 6e-16)):
        p = tab[s, deg, m]
        for k in range(deg - 1, -1, -1):
            p = (p.astype(ld) * v.astype(ld) + tab[s, k, m].astype(ld)).astype(float)
        err = p - want[:, m]
        if m:
            err = err / want[:, m]
        got = float(np.sqrt((err ** 2).mean())), float(np.abs(err).max())
        print(f"{name}: rms {got[0]:.2e} worst {got[1]:.2e}")
        assert got[0] < rms and got[1] < worst, (name, got)
