"""The generators' half-space passes at the sizes where they can go wrong --
the smallest box, odd numbers of z lines (the variance ends inside a line),
axes at and beyond the passes' LDS bounds, mixed-radix and Bluestein lengths
on each axis -- element-wise against the CPU oracle on the same Philox
stream.  The bound is the generators' own 1e-11 relative L2: the passes sum
in another order than the oracle, FP64 throughout (1e-15 to 1e-14 seen)."""
import numpy as np
import pytest

from hammurabix_amd import _capi as capi
from hammurabix_amd.units import CGS
from oracle_lib import load_oracle, ptr, rel_l2
import ctypes as C

pytestmark = pytest.mark.gpu

SHAPES = [(2, 2, 2), (3, 5, 7), (16, 8, 4), (33, 17, 9), (64, 48, 128), (11, 26, 13),
          (5, 3, 37),
          (4, 6, 1024), (3, 2, 512),    # z at the passes' bound
          (4, 3, 1100), (2, 2, 1031),   # ... and beyond it: whole-array steps
          (2100, 3, 2), (4096, 2, 3),   # x in the largest tile
          (1031, 3, 2),                 # Bluestein x of 4096 points
          (4116, 2, 2), (2053, 2, 2)]   # x beyond the bound


def box(shape):
    return capi.HamxBox(*shape, -20 * CGS.kpc, 20 * CGS.kpc, -20 * CGS.kpc, 20 * CGS.kpc,
                        -4 * CGS.kpc, 4 * CGS.kpc)


def fill(d, shape):
    d.box = box(shape)
    d.observer[:] = [-8.3 * CGS.kpc, 0.0, 0.006 * CGS.kpc]
    if hasattr(d, "breg_model"):
        d.breg_model = capi.HAMX_BREG_LSA
        d.breg[0:4] = [6e-6, 27 * CGS.rad, 0.9 * CGS.rad, 25 * CGS.rad]
    return d


def compare(gpu, oracle, d, seed, shape, outs, bound=1e-11):
    n = int(np.prod(shape))
    g = [np.full(n, np.nan) for _ in range(outs)]
    r = [np.zeros(n) for _ in range(outs)]
    gpu(d, seed, *g)
    assert oracle(C.byref(d), seed, *[ptr(a) for a in r]) == 0
    for a, b in zip(g, r):
        assert np.all(np.isfinite(a))
        assert rel_l2(a, b) < bound


def es(shape, rho):
    d = fill(capi.HamxEsDesc(), shape)
    d.rms, d.k0, d.k1, d.a0, d.a1, d.rho = 2e-6, 0.12, 0.06, 1.7, 0.5, rho
    d.r0, d.z0 = 8 * CGS.kpc, 1 * CGS.kpc
    return d


@pytest.mark.parametrize("shape", SHAPES)
def test_es(ctx, shape):
    compare(ctx.brnd_es, load_oracle().orc_brnd_es, es(shape, 0.7), 5, shape, 3)


@pytest.mark.parametrize("shape", SHAPES)
def test_dft(ctx, shape):
    d = fill(capi.HamxDftDesc(), shape)
    d.rms, d.k0, d.a0, d.r0, d.z0 = 1e-3, 0.02, -1.7, 8 * CGS.kpc, 1 * CGS.kpc
    compare(ctx.ternd_dft, load_oracle().orc_ternd_dft, d, 6, shape, 1)


@pytest.mark.parametrize("z0", [1.0, 0.009])  # 0.009 kpc: the profile is not split
@pytest.mark.parametrize("model", ["helix", "none", "lsa_off", "jf12_profile"])
def test_rescale_routes(ctx, model, z0):
    shape = (20, 18, 12)
    d = es(shape, 1.6)
    d.z0 = z0 * CGS.kpc
    orc = load_oracle()
    if model == "helix":  # zero field outside 5-15 kpc: raw values there
        d.breg_model = capi.HAMX_BREG_HELIX
        d.breg[0:5] = [1e-6, 2e-6, 0.5e-6, 5 * CGS.kpc, 15 * CGS.kpc]
    elif model == "none":
        d.breg_model = capi.HAMX_BREG_NONE
    elif model == "lsa_off":
        d.breg[0] = 0.0
    if model == "jf12_profile":
        mu, kpc = 1e-6, CGS.kpc
        d.jf12[:] = [10.81 * mu, 6.96 * mu, 9.59 * mu, 6.96 * mu, 1.96 * mu, 16.34 * mu,
                     37.29 * mu, 10.35 * mu, 7.63 * mu, 0.61 * kpc, 4.68 * mu, 10.97 * kpc,
                     2.84 * kpc]
        compare(ctx.brnd_jf12, orc.orc_brnd_jf12, d, 5, shape, 3)
    else:
        compare(ctx.brnd_es, orc.orc_brnd_es, d, 5, shape, 3)


@pytest.mark.parametrize("z0", [1.0, 0.009])
def test_dft_profile_routes(ctx, z0):
    shape = (20, 18, 12)
    d = fill(capi.HamxDftDesc(), shape)
    d.rms, d.k0, d.a0, d.r0, d.z0 = 1e-3, 0.02, -1.7, 8 * CGS.kpc, z0 * CGS.kpc
    compare(ctx.ternd_dft, load_oracle().orc_ternd_dft, d, 6, shape, 1)


def mhd(shape):
    d = fill(capi.HamxMhdDesc(), shape)
    d.pa0 = d.pf0 = d.ps0 = 1e-12
    d.k0, d.k1, d.aa0, d.af0, d.as0, d.a1, d.beta, d.ma = 0.3, 0.1, 1.7, 1.5, 1.7, 0.0, 0.1, 0.5
    return d


@pytest.mark.parametrize("shape", SHAPES)
def test_mhd(ctx, shape):
    compare(ctx.brnd_mhd, load_oracle().orc_brnd_mhd, mhd(shape), 7, shape, 3)


# Wave numbers beyond half of an axis carry the rounding of n/L: on an axis of
# 4096 points the lowest negative one is 5e-13 off its mirror, and 2e-14 or more
# in the field if one of the pair stands for both.  With each mode's own only the
# rounding of the sums is left: three transforms of 2^-53 log2(n) and the models'
# few ulps, below 3e-15 on either side.
WAVE = [(4096, 4, 6), (6, 4000, 4), (4, 6, 1000)]


@pytest.mark.parametrize("shape", WAVE)
def test_es_takes_each_wave_vector(ctx, shape):
    print("case: es wave vectors", shape, flush=True)
    compare(ctx.brnd_es, load_oracle().orc_brnd_es, es(shape, 1.3), 5, shape, 3, bound=6e-15)


@pytest.mark.parametrize("shape", WAVE)
def test_mhd_takes_each_wave_vector(ctx, shape):
    print("case: mhd wave vectors", shape, flush=True)
    compare(ctx.brnd_mhd, load_oracle().orc_brnd_mhd, mhd(shape), 5, shape, 3, bound=6e-15)


@pytest.mark.parametrize("gen", ["es", "dft", "mhd"])
def test_spectra_far_from_one_per_kpc(ctx, gen):
    """Spectra of boxes 1e20 times as large: |k| enters relative to k0, so the
    rounding of its logarithm (1.4e-14 once multiplied by the exponent, were it
    taken in 1/kpc) leaves the sums' 3e-15 alone."""
    shape, big = (24, 20, 16), 1e20
    orc = load_oracle()
    if gen == "es":
        d = es(shape, 1.0)
        d.k0, d.k1, d.a0, d.a1 = 0.12 / big, 0.06 / big, 3.7, 0.5
        call, ref, outs = ctx.brnd_es, orc.orc_brnd_es, 3
    elif gen == "dft":
        d = fill(capi.HamxDftDesc(), shape)
        d.rms, d.k0, d.a0, d.r0, d.z0 = 1e-3, 0.02 / big, -3.7, 8 * CGS.kpc, 1 * CGS.kpc
        call, ref, outs = ctx.ternd_dft, orc.orc_ternd_dft, 1
    else:
        d = mhd(shape)
        d.k0, d.k1, d.aa0, d.af0, d.as0 = 0.3 / big, 0.1 / big, 3.7, 3.5, 3.7
        call, ref, outs = ctx.brnd_mhd, orc.orc_brnd_mhd, 3
    for f in ("x_min", "x_max", "y_min", "y_max", "z_min", "z_max"):
        setattr(d.box, f, getattr(d.box, f) * big)
    if gen != "mhd":
        d.r0, d.z0 = d.r0 * big, d.z0 * big
    compare(call, ref, d, 8, shape, outs, bound=6e-15)


@pytest.mark.parametrize("half", [True, False])
@pytest.mark.parametrize("tilt", [0.0, 3e-7, 3e-6])
def test_mhd_along_the_field(ctx, tilt, half):
    """Modes along a regular field that is off the z axis by less than 1e-6 (their
    versors' small components stay), exactly on it, or by enough to count as
    across it; half-space passes and whole-array steps."""
    shape = (6, 4, 10) if half else (3, 2, 1100)
    d = mhd(shape)
    d.breg_model = capi.HAMX_BREG_CART
    d.breg[0:3] = [tilt * 2e-6, -0.4 * tilt * 2e-6, 2e-6]
    compare(ctx.brnd_mhd, load_oracle().orc_brnd_mhd, d, 9, shape, 3)


def test_mhd_modes_without_power(ctx):
    """A fast mode whose h_f is 0 stays exactly 0, however large its norm (here
    every one, by a plasma beta without an h_f; sqrt(norm) = 1e150)."""
    d = mhd((12, 10, 8))
    d.beta, d.pf0 = np.nan, 1e300
    compare(ctx.brnd_mhd, load_oracle().orc_brnd_mhd, d, 10, (12, 10, 8), 3)
