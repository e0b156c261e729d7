"""The specialised march with every regular-field and electron model, with
and without packed random grids, for a spectral index of 3 (emissivity as a
product) and 2.8 (as a power), on the default schedule against the CPU
oracle: FP64 maps within 1e-10 relative L2 (the plain-path bar)."""
import numpy as np
import pytest

from hammurabix_amd import HamxError, Param, _capi as capi, configs
from hammurabix_amd.units import CGS
from oracle_lib import write_grid
from test_gpu_los import assert_parity, gpu_maps, random_grids
from test_oracle_models import jf12_params

pytestmark = pytest.mark.gpu


def set_breg(d, name):
    mu, kpc = 1e-6, CGS.kpc
    if name == "none":
        d.breg_model = capi.HAMX_BREG_NONE
    elif name == "cart":
        d.breg_model = capi.HAMX_BREG_CART
        d.breg[0:3] = [1 * mu, 2 * mu, 0.5 * mu]
    elif name == "helix":
        d.breg_model = capi.HAMX_BREG_HELIX
        d.breg[0:5] = [1 * mu, 2 * mu, 0.5 * mu, 3 * kpc, 12 * kpc]
    elif name == "jf12":
        d.breg_model = capi.HAMX_BREG_JF12
        d.breg[0:20] = list(jf12_params())
    elif name == "grid":
        d.breg_model = capi.HAMX_BREG_GRID


MODELS = [("none", "unif"), ("cart", "none"), ("helix", "unif"), ("grid", "grid"), ("lsa", "none"),
          ("lsa", "ymw16"), ("cart", "ymw16"), ("jf12", "unif"), ("jf12", "ymw16")]


def check_models(ctx, breg, tereg, random, alpha, **kw):
    par = Param(text=configs.random_forward(
        grid=(16, 16, 8), tereg="ymw16" if tereg == "ymw16" else "unif", **kw))
    d = par.los_desc()
    d.cre[0] = alpha
    set_breg(d, breg)
    grids = {}
    b, te, box = random_grids((16, 16, 8), seed=3, te_scale=0.002)
    if random:
        grids.update(brnd=b, brnd_box=box, ternd=te, ternd_box=box)
    if breg == "grid":
        g, t, gbox = random_grids((9, 11, 7), seed=4)
        grids.update(breg=g, breg_box=gbox, tereg=np.abs(t), tereg_box=gbox)
    if tereg == "grid":
        d.tereg_model = capi.HAMX_TEREG_GRID
    elif tereg == "none":
        d.tereg_model = capi.HAMX_TEREG_NONE
    if (breg, random) == ("none", False):
        pytest.skip("no field at all: nothing to compare")
    if tereg == "none" and not random:
        d.do_dm = d.do_fd = 0  # zero maps
    ref = {k: v for k, v in write_grid(d, **grids).items() if np.any(v)}
    got = gpu_maps(ctx, d, **grids)
    assert_parity({k: got[k] for k in ref}, ref, label=f"{breg}/{tereg}")


@pytest.mark.parametrize("alpha", [3.0, 2.8])
@pytest.mark.parametrize("random", [True, False])
@pytest.mark.parametrize("breg,tereg", MODELS)
def test_models(ctx, breg, tereg, random, alpha):
    """Small shells: four wavefronts on a ray."""
    print("case:", breg, tereg, random, alpha, flush=True)
    check_models(ctx, breg, tereg, random, alpha, nside_sim=2, nside_out=8, oc_r_res=0.043)


@pytest.mark.parametrize("alpha", [3.0, 2.8])
@pytest.mark.parametrize("random", [True, False])
@pytest.mark.parametrize("breg,tereg", MODELS)
def test_models_on_large_shells(ctx, breg, tereg, random, alpha):
    """Shells from nside 32 on: a wavefront marches two rays in turn."""
    print("case: large", breg, tereg, random, alpha, flush=True)
    check_models(ctx, breg, tereg, random, alpha, shell_num=2, nside_sim=32, nside_out=32,
                 oc_r_res=0.17)


def test_ymw16_through_its_nebulae(ctx):
    """A short, finely sampled shell about the Sun: the Local Bubble, Loop I
    and the Gum shell, whose shortened forms are this march's own."""
    par = Param(text=configs.plain_forward(tereg="ymw16", nside_sim=8, nside_out=8,
                                           oc_r_max=1.5, oc_r_res=0.002))
    d = par.los_desc()
    assert_parity(gpu_maps(ctx, d), write_grid(d), label="ymw16 nebulae")


def ymw16_near(schedule=capi.HAMX_SCHED_AUTO):
    """Rays through the nebulae about the Sun and the disks to 12 kpc."""
    return Param(text=configs.plain_forward(tereg="ymw16", shell_num=2, nside_sim=4, nside_out=4,
                                            oc_r_max=12., oc_r_res=0.03)).los_desc(schedule=schedule)


def compare_ymw16(ctx, d, label):
    """Parity with the oracle, or refused where its maps are not finite."""
    with np.errstate(all="ignore"):
        ref = write_grid(d)
    print("case:", label, flush=True)
    if all(np.all(np.isfinite(v)) for v in ref.values()):
        assert_parity(gpu_maps(ctx, d), ref, label=label)
    else:
        with pytest.raises(HamxError, match="non-finite"):
            gpu_maps(ctx, d)


# the scale lengths and angular widths of every component
YMW16_SCALES = [3, 6, 7, 10, 17, 18, 19, 20, 42, 43, 46, 49, 51, 52, 54, 60, 61, 62, 65, 66, 67,
                70, 71]


@pytest.mark.parametrize("sched", [capi.HAMX_SCHED_AUTO, capi.HAMX_SCHED_WAVE])
@pytest.mark.parametrize("value", [0.0, 1.0, "negative"])
def test_ymw16_scales_out_of_range(ctx, value, sched):
    """A scale of 0 (or 1 cm, 1 degree) turns its component off, wholly or off
    its own surface; a negative one is its magnitude within its sech^2."""
    for i in YMW16_SCALES:
        d = ymw16_near(sched)
        d.tereg[i] = -d.tereg[i] if value == "negative" else value
        compare_ymw16(ctx, d, f"ymw16 scale {i} = {value}")


@pytest.mark.parametrize("sched", [capi.HAMX_SCHED_AUTO, capi.HAMX_SCHED_WAVE])
def test_ymw16_arm_across_the_circle(ctx, sched):
    """Pitch angles to a right angle."""
    for pitch in (np.pi / 2, -np.pi / 2, 1.5707, 1.4):
        d = ymw16_near(sched)
        d.tereg[32], d.tereg[37] = np.tan(pitch), np.cos(pitch)
        compare_ymw16(ctx, d, f"ymw16 pitch {pitch}")
    d = ymw16_near(sched)
    d.tereg[37] = -d.tereg[37]  # the distance from the arm changes sign
    compare_ymw16(ctx, d, "ymw16 negative cosine")
    d = ymw16_near(sched)
    d.tereg[27] = -1e7
    compare_ymw16(ctx, d, "ymw16 arm out of reach")


@pytest.mark.parametrize("sched", [capi.HAMX_SCHED_AUTO, capi.HAMX_SCHED_WAVE])
@pytest.mark.parametrize("n1", [0.0, 0.01])
def test_ymw16_bubble_without_disks(ctx, n1, sched):
    """Where the disks are 0 any bubble term above 0 decides, here 1e-60 and
    less against a wide Loop I above a thick disk of 20 pc."""
    d = ymw16_near(sched)
    d.tereg[5], d.tereg[6] = n1, 20 * CGS.pc
    d.tereg[9] = 0.0
    for i in range(12, 17):
        d.tereg[i] = 0.0
    for i in (61, 62, 66, 67):
        d.tereg[i] = 1.3 * CGS.pc
    d.tereg[70], d.tereg[71] = 100 * CGS.pc, 300.0
    compare_ymw16(ctx, d, "ymw16 bubble without disks")


@pytest.mark.parametrize("value", [np.nan, np.inf])
def test_ymw16_parameter_not_finite(ctx, value):
    """Refused where the model's own weighting (0 times what is not chosen)
    makes the density NaN, accepted where it does not.  (The disk's and the arms'
    NaN is left out: the oracle takes the larger of the two by std::max, which
    drops the other one.)"""
    disk = range(7, 50) if np.isnan(value) else range(44, 50)
    for i in sorted(set(range(73)) - set(disk) - {0, 3, 4, 50, 52}):
        d = ymw16_near()
        d.tereg[i] = value
        compare_ymw16(ctx, d, f"ymw16 parameter {i} = {value}")


@pytest.mark.parametrize("sched", [capi.HAMX_SCHED_AUTO, capi.HAMX_SCHED_WAVE])
def test_ymw16_gum_shell_out_of_range(ctx, sched):
    """A Gum shell without radius, inside out or flattened beyond measure."""
    for a, k in ((0.0, 1.0), (1.0, -1.4), (-1.0, 1.4), (1.0, 0.0), (1e-80, 1.4)):
        d = ymw16_near(sched)
        d.tereg[55], d.tereg[56] = a * d.tereg[55], k
        compare_ymw16(ctx, d, f"ymw16 gum shell {a} {k}")


@pytest.mark.parametrize("sched", [capi.HAMX_SCHED_AUTO, capi.HAMX_SCHED_WAVE])
@pytest.mark.parametrize("breg", ["cart", "lsa"])
@pytest.mark.parametrize("what", ["r_min", "r_max", "te", "cre"])
def test_negative_limits(ctx, what, breg, sched):
    """No length is below a negative lower limit; every one is above a negative
    radius (the specialised march compares squares)."""
    print("case: negative", what, breg, sched, flush=True)
    d = Param(text=configs.plain_forward(nside_sim=2, nside_out=2, oc_r_res=0.1)).los_desc(
        schedule=sched)
    set_breg(d, breg)
    if what == "r_min":
        d.gc_r_min = -12 * CGS.kpc
    elif what == "r_max":
        d.gc_r_max = -12 * CGS.kpc
    elif what == "te":
        d.tereg[1] = -6 * CGS.kpc
    else:
        d.cre_model = capi.HAMX_CRE_UNIF
        d.cre[0:4] = [3.0, -6 * CGS.kpc, 20.6 * CGS.GeV, 0.0217]
    ref, got = write_grid(d), gpu_maps(ctx, d)
    zero = {k for k, v in ref.items() if not np.any(v)}
    assert zero == {"r_min": set(), "r_max": set(ref), "te": {"dm", "fd"},
                    "cre": {"is", "qs", "us"}}[what]
    assert not any(np.any(got[k]) for k in zero)
    assert_parity({k: got[k] for k in ref if k not in zero},
                  {k: ref[k] for k in ref if k not in zero}, label=f"negative {what}")
