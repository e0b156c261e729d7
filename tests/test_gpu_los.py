"""GPU parity of the LOS integrator (hamx_los_forward) against the CPU
oracle: FP64 maps within 1e-10 relative L2 per map (the plain-path bar),
both march schedules, grids gathered packed and separate, FD carried
across shells, outputs accumulated across nside, and the error paths.
"""
import math

import numpy as np
import pytest

from hammurabix_amd import HamxError, Param, _capi as capi, configs
from hammurabix_amd.units import CGS
from oracle_lib import fields_struct, npix, rel_l2, write_grid

pytestmark = pytest.mark.gpu

TOL = 1e-10  # relative L2 per map, FP64 plain path
MAPS = ("dm", "fd", "is", "qs", "us")


def gpu_maps(ctx, desc, **grids):
    m = {}
    if desc.do_dm:
        m["dm"] = np.zeros(npix(desc.nside_dm))
    if desc.do_sync:
        for k in ("is", "qs", "us"):
            m[k] = np.zeros(npix(desc.nside_sync))
    if desc.do_fd or desc.do_sync:
        m["fd"] = np.zeros(npix(desc.nside_fd if desc.do_fd else desc.nside_sync))
    ctx.los_forward(desc, m, **grids)
    return m


def assert_parity(got, ref, tol=TOL, label=""):
    assert set(got) == set(ref)
    for k in ref:
        err = rel_l2(got[k], ref[k])
        print(f"{label} {k}: rel L2 {err:.3e}", flush=True)
        assert np.all(np.isfinite(got[k])), k
        assert err <= tol, f"{label} map {k}: rel L2 {err:.3e} > {tol}"


def random_grids(shape, seed=0, te_scale=0.003):
    rng = np.random.default_rng(seed)
    n = int(np.prod(shape))
    b = tuple(np.ascontiguousarray(rng.normal(0, 2e-6, n)) for _ in range(3))
    te = np.ascontiguousarray(rng.normal(0.0, te_scale, n))  # negative values hit the clamp
    box = capi.HamxBox(*shape, -20 * CGS.kpc, 20 * CGS.kpc, -20 * CGS.kpc, 20 * CGS.kpc,
                       -4 * CGS.kpc, 4 * CGS.kpc)
    return b, te, box


@pytest.mark.parametrize("sched", [capi.HAMX_SCHED_THREAD, capi.HAMX_SCHED_WAVE,
                                   capi.HAMX_SCHED_AUTO])
def test_plain_forward_full_size(ctx, sched):
    """LSA + uniform TE + analytic CRE, one shell at nside 32, 3000 steps."""
    print("case: plain forward nside 32, schedule", sched, flush=True)
    par = Param(text=configs.plain_forward())
    d = par.los_desc(schedule=sched)
    assert_parity(gpu_maps(ctx, d), write_grid(d), label=f"plain/{sched}")


@pytest.mark.parametrize("sched", [capi.HAMX_SCHED_THREAD, capi.HAMX_SCHED_WAVE,
                                   capi.HAMX_SCHED_AUTO])
@pytest.mark.parametrize("packed", [True, False])
def test_random_grids_multishell(ctx, sched, packed):
    """3 shells (8/16/32), brnd + ternd grids, FD carried through the shells."""
    print("case: multishell grids, schedule", sched, "packed", packed, flush=True)
    par = Param(text=configs.random_forward(nside_sim=8, nside_out=32, oc_r_res=0.05,
                                            grid=(32, 32, 16)))
    d = par.los_desc(schedule=sched)
    b, te, box = random_grids((32, 32, 16))
    ternd_box = box
    if not packed:  # a different TE box forces the separate gathers
        ternd_box = capi.HamxBox(32, 32, 16, -21 * CGS.kpc, 19 * CGS.kpc, -20 * CGS.kpc,
                                 20 * CGS.kpc, -4 * CGS.kpc, 4 * CGS.kpc)
    ref = write_grid(d, brnd=b, brnd_box=box, ternd=te, ternd_box=ternd_box)
    got = gpu_maps(ctx, d, brnd=b, brnd_box=box, ternd=te, ternd_box=ternd_box)
    assert_parity(got, ref, label=f"grids/{sched}/{packed}")


def test_output_nsides_differ_from_shells(ctx):
    """DM at nside 16, FD at 64, sync at 8: every accumulate interpolates."""
    par = Param(text=configs.random_forward(nside_sim=8, nside_out=32, oc_r_res=0.05,
                                            grid=(32, 32, 16)))
    d = par.los_desc()
    d.nside_dm, d.nside_fd, d.nside_sync = 16, 64, 8
    b, te, box = random_grids((32, 32, 16), seed=4)
    ref = write_grid(d, brnd=b, brnd_box=box, ternd=te, ternd_box=box)
    got = gpu_maps(ctx, d, brnd=b, brnd_box=box, ternd=te, ternd_box=box)
    assert_parity(got, ref, label="nsides")


@pytest.mark.parametrize("flags", [(1, 0, 0), (0, 1, 0), (0, 0, 1), (1, 0, 1), (0, 1, 1)])
def test_observable_subsets(ctx, flags):
    """Only DM, only FD, only sync (zero FD cache), and mixtures."""
    par = Param(text=configs.random_forward(nside_sim=4, nside_out=16, oc_r_res=0.1,
                                            grid=(16, 16, 8)))
    d = par.los_desc()
    d.do_dm, d.do_fd, d.do_sync = flags
    b, te, box = random_grids((16, 16, 8), seed=5)
    ref = write_grid(d, brnd=b, brnd_box=box, ternd=te, ternd_box=box)
    got = gpu_maps(ctx, d, brnd=b, brnd_box=box, ternd=te, ternd_box=box)
    assert_parity(got, ref, label=f"subset{flags}")


def test_regular_field_grids_and_variable_cre_index(ctx):
    """Imported breg/tereg grids (HAMX_BREG_GRID / HAMX_TEREG_GRID) and a CRE
    spectral index varying with r and z (Gamma factors on the device)."""
    par = Param(text=configs.plain_forward(nside_sim=8, nside_out=8, oc_r_res=0.05))
    d = par.los_desc()
    b, te, box = random_grids((24, 24, 12), seed=6, te_scale=0.01)
    d.breg_model = capi.HAMX_BREG_GRID
    d.tereg_model = capi.HAMX_TEREG_GRID
    d.cre[1] = 0.02  # beta
    d.cre[2] = 0.05  # theta
    te_pos = np.abs(te)
    ref = write_grid(d, breg=b, breg_box=box, tereg=te_pos, tereg_box=box)
    got = gpu_maps(ctx, d, breg=b, breg_box=box, tereg=te_pos, tereg_box=box)
    assert_parity(got, ref, tol=1e-9, label="breg-grid")  # Lanczos Gamma ~1e-14


@pytest.mark.parametrize("model", [capi.HAMX_BREG_CART, capi.HAMX_BREG_UNIF])
def test_cart_unif_models_with_cre_unif(ctx, model):
    par = Param(text=configs.plain_forward(nside_sim=4, nside_out=4, oc_r_res=0.05))
    d = par.los_desc()
    d.breg_model = model
    d.breg[0:3] = [1.5e-6, -2e-6, 0.6] if model == capi.HAMX_BREG_UNIF else [1.5e-6, -2e-6, 7e-7]
    d.cre_model = capi.HAMX_CRE_UNIF
    d.cre[0:4] = [3.0, 4 * CGS.kpc, 20.6 * CGS.GeV, 0.0217]
    assert_parity(gpu_maps(ctx, d), write_grid(d), label=f"model{model}")


@pytest.mark.parametrize("model,variant", [(capi.HAMX_BREG_HELIX, ""), (capi.HAMX_BREG_JF12, ""),
                                           (capi.HAMX_BREG_JAFFE, "bar"),
                                           (capi.HAMX_BREG_JAFFE, "ring")])
def test_helix_jf12_jaffe_models(ctx, model, variant):
    """The helix, JF12 and Jaffe regular fields on the device against the
    oracle's restatements (breg_helix.cc:13-30, breg_jf12.cc:8-189,
    breg_jaffe.cc:11-243), with random grids added, at the template's
    parameters (Jaffe also with the ring, quadruple and bss)."""
    from test_oracle_models import jaffe_params, jf12_params
    print(f"case: breg model {model} {variant}", flush=True)
    par = Param(text=configs.random_forward(nside_sim=4, nside_out=8, oc_r_res=0.05,
                                            grid=(16, 16, 8)))
    d = par.los_desc()
    d.breg_model = model
    if model == capi.HAMX_BREG_HELIX:
        d.breg[0:5] = [1e-6, 2e-6, 0.5e-6, 3 * CGS.kpc, 12 * CGS.kpc]
    elif model == capi.HAMX_BREG_JF12:
        d.breg[0:20] = list(jf12_params())
    else:
        over = dict(ring=1.0, bar=0.0, quadruple=1.0, bss=1.0) if variant == "ring" else {}
        d.breg[0:33] = list(jaffe_params(**over))
    b, te, box = random_grids((16, 16, 8), seed=12)
    kw = dict(brnd=b, brnd_box=box, ternd=te, ternd_box=box)
    assert_parity(gpu_maps(ctx, d, **kw), write_grid(d, **kw), label=f"model{model}")


@pytest.mark.parametrize("sched", [capi.HAMX_SCHED_WAVE, capi.HAMX_SCHED_THREAD])
@pytest.mark.parametrize("breg", ["lsa", "jf12"])
def test_ymw16_thermal_electrons(ctx, sched, breg):
    """YMW16 (tereg_ymw16.cc:10-333) at the template's parameters on the
    device against the oracle's restatement, with random grids added; DM
    probes the density directly, FD and the Faraday-rotated Q/U through B."""
    from test_oracle_models import jf12_params
    print(f"case: ymw16 schedule {sched} breg {breg}", flush=True)
    par = Param(text=configs.random_forward(nside_sim=4, nside_out=8, oc_r_res=0.05,
                                            grid=(16, 16, 8), tereg="ymw16"))
    d = par.los_desc(schedule=sched)
    assert d.tereg_model == capi.HAMX_TEREG_YMW16
    if breg == "jf12":
        d.breg_model = capi.HAMX_BREG_JF12
        d.breg[0:20] = list(jf12_params())
    b, te, box = random_grids((16, 16, 8), seed=13, te_scale=0.0003)
    kw = dict(brnd=b, brnd_box=box, ternd=te, ternd_box=box)
    ref = write_grid(d, **kw)
    assert np.linalg.norm(ref["dm"]) > 0
    assert_parity(gpu_maps(ctx, d, **kw), ref, label=f"ymw16/{sched}/{breg}")


def test_empty_shell_and_no_samples(ctx):
    """A shell thinner than one step contributes nothing; so does a sky with
    every sample outside the galactocentric limits."""
    par = Param(text=configs.plain_forward(nside_sim=4, nside_out=4, oc_r_res=0.05))
    d = par.los_desc()
    d.n_shell = 2
    d.nside_shell[1] = 8
    d.radii_shell[1] = 0.01 * CGS.kpc
    d.radii_shell[2] = 30 * CGS.kpc
    assert_parity(gpu_maps(ctx, d), write_grid(d), label="empty-shell")
    d.gc_r_max = 1.0 * CGS.kpc  # observer sits 8.3 kpc out: no sample passes
    got = gpu_maps(ctx, d)
    for k in got:
        assert np.all(got[k] == 0.0)


def test_device_resident_buffers(ctx):
    """Torch device tensors in and out (HAMX_IN_DEVICE | HAMX_OUT_DEVICE)."""
    import torch
    par = Param(text=configs.random_forward(nside_sim=4, nside_out=16, oc_r_res=0.1,
                                            grid=(16, 16, 8)))
    d = par.los_desc()
    b, te, box = random_grids((16, 16, 8), seed=8)
    ref = write_grid(d, brnd=b, brnd_box=box, ternd=te, ternd_box=box)
    db = tuple(torch.from_numpy(a).cuda() for a in b)
    dte = torch.from_numpy(te).cuda()
    m = {k: torch.zeros(v.shape[0], dtype=torch.float64, device="cuda") for k, v in ref.items()}
    ctx.los_forward(d, m, brnd=db, brnd_box=box, ternd=dte, ternd_box=box)
    assert_parity({k: v.cpu().numpy() for k, v in m.items()}, ref, label="device")


def test_errors_are_reported(ctx):
    par = Param(text=configs.plain_forward(nside_sim=4, nside_out=4))
    d = par.los_desc()
    d.nside_shell[0] = 6
    with pytest.raises(HamxError) as e:
        gpu_maps(ctx, d)
    assert e.value.code == capi.HAMX_ERR_NSIDE
    d = par.los_desc()
    d.cre_model = capi.HAMX_CRE_NONE
    with pytest.raises(HamxError) as e:
        gpu_maps(ctx, d)
    assert e.value.code == capi.HAMX_ERR_ARG
    assert "CRE" in str(e.value)
    # the context stays usable after an error
    d = par.los_desc()
    assert_parity(gpu_maps(ctx, d), write_grid(d), label="after-error")


def test_uniform_sphere_closed_form_on_device(ctx):
    """Same closed form as the oracle test, evaluated on the device path."""
    d = capi.HamxLosDesc()
    nside, r0, res, rmax, freq = 2, 2.0, 0.013, 3.0, 1.4e9
    B = np.array([1.5e-6, -2.0e-6, 0.7e-6])
    d.n_shell = 1
    d.nside_shell[0] = nside
    d.radii_shell[1] = rmax * CGS.kpc
    d.oc_r_res = res * CGS.kpc
    d.gc_r_max = 1e3 * CGS.kpc
    d.gc_z_min, d.gc_z_max = -1e3 * CGS.kpc, 1e3 * CGS.kpc
    d.do_dm = d.do_fd = d.do_sync = 1
    d.nside_dm = d.nside_fd = d.nside_sync = nside
    d.sync_freq = freq
    d.breg_model = capi.HAMX_BREG_CART
    d.breg[0:3] = B
    d.tereg_model = capi.HAMX_TEREG_UNIF
    d.tereg[0:2] = [0.02, r0 * CGS.kpc]
    d.cre_model = capi.HAMX_CRE_UNIF
    d.cre[0:4] = [3.0, r0 * CGS.kpc, 20.6 * CGS.GeV, 0.0217]
    got = gpu_maps(ctx, d)
    step = math.floor(rmax / res)
    delta = rmax * CGS.kpc / step
    K = int(np.sum((np.arange(step) + 0.5) * delta <= r0 * CGS.kpc))
    np.testing.assert_allclose(got["dm"], 0.02 * K * delta, rtol=1e-12)


def test_masked_pass_matches_oracle(ctx):
    """The reference's nside-8 mask fixture over shells at nside 4/8/16 (the
    mask is downgraded, used as is, and upgraded), random grids, FD carry."""
    import os
    print("case: masked multishell", flush=True)
    piv = np.ascontiguousarray(np.fromfile(
        os.path.join(os.path.dirname(__file__), "golden", "mask_map_nside8.bin"), dtype="<f8"))
    par = Param(text=configs.random_forward(nside_sim=4, nside_out=16, oc_r_res=0.05,
                                            grid=(32, 32, 16)))
    d = par.los_desc()
    b, te, box = random_grids((32, 32, 16), seed=9)
    kw = dict(brnd=b, brnd_box=box, ternd=te, ternd_box=box)
    ref = write_grid(d, mask=piv, nside_mask=8, **kw)
    m = {k: np.zeros_like(v) for k, v in ref.items()}
    ctx.los_forward(d, m, mask=piv, nside_mask=8, **kw)
    assert_parity(m, ref, label="masked")
    full = write_grid(d, **kw)
    assert any(rel_l2(ref[k], full[k]) > 1e-3 for k in ref)  # the mask matters


@pytest.mark.parametrize("where", ["brnd", "ternd"])
def test_nan_in_a_grid_is_an_error(ctx, where):
    """A NaN in an input grid (the reference's debug build asserts isfinite on
    B_par, B_per, te and the phase, integrator.cc:192,195,202,223) comes back
    as an error naming the non-finite values; the context stays usable."""
    par = Param(text=configs.random_forward(nside_sim=4, nside_out=8, oc_r_res=0.1,
                                            grid=(16, 16, 8)))
    d = par.los_desc()
    b, te, box = random_grids((16, 16, 8), seed=21)
    bad_b = tuple(a.copy() for a in b)
    bad_te = te.copy()
    # a vertex near the observer, inside the box, that the rays sample
    v = (5 * 16 + 8) * 8 + 4
    if where == "brnd":
        bad_b[1][v] = np.nan
    else:
        bad_te[v] = np.nan
    with pytest.raises(HamxError) as e:
        gpu_maps(ctx, d, brnd=bad_b, brnd_box=box, ternd=bad_te, ternd_box=box)
    assert e.value.code == capi.HAMX_ERR_ARG and "non-finite" in str(e.value)
    assert_parity(gpu_maps(ctx, d, brnd=b, brnd_box=box, ternd=te, ternd_box=box),
                  write_grid(d, brnd=b, brnd_box=box, ternd=te, ternd_box=box), label="after-nan")


def test_phase_rotation_beyond_the_reduced_range(ctx):
    """At 3 MHz (lambda^2 = 1e4 m^2) the Faraday phase 2 lambda^2 FD of the
    outer samples exceeds 2^19 pi, where the march's Cody-Waite reduction
    hands over to the library sine and cosine; the inner ones stay below it.
    DM, FD and I at the plain-path bar; Q and U at 1e-6: an FD summed in
    another order differs by ~1e-15 relative, which moves a phase of millions
    of radians by ~1e-9 (a wrong sine or cosine would be off by O(1))."""
    print("case: Faraday phase beyond 2^19 pi", flush=True)
    par = Param(text=configs.plain_forward(nside_sim=8, nside_out=8, oc_r_res=0.05))
    d = par.los_desc()
    d.sync_freq = 3e6
    got, ref = gpu_maps(ctx, d), write_grid(d)
    lam2 = (CGS.c_light / d.sync_freq) ** 2  # cm^2; the raw FD map is per cm^2
    big = np.abs(2 * lam2 * ref["fd"]).max()
    print(f"largest shell-end phase {big:.3e} rad (reduction limit {2**19 * math.pi:.3e})",
          flush=True)
    assert big > 2 ** 19 * math.pi
    assert_parity({k: got[k] for k in ("dm", "fd", "is")}, {k: ref[k] for k in ("dm", "fd", "is")},
                  label="3 MHz")
    assert_parity({k: got[k] for k in ("qs", "us")}, {k: ref[k] for k in ("qs", "us")}, tol=1e-6,
                  label="3 MHz")


@pytest.mark.parametrize("angles", [(60.0, 25.0), (27.0, 70.0), (-100.0, -50.0)])
def test_lsa_angles_beyond_a_quarter_turn(ctx, angles):
    """psi0 or chi0 beyond 45 degrees: psi(r), chi(z) leave [-pi/4, pi/4], so
    the LSA's sines and cosines take the library path instead of the series."""
    psi0, chi0 = angles
    print(f"case: LSA psi0 {psi0} chi0 {chi0} degrees", flush=True)
    par = Param(text=configs.plain_forward(nside_sim=8, nside_out=8, oc_r_res=0.05))
    d = par.los_desc()
    d.breg[1] = math.radians(psi0)
    d.breg[3] = math.radians(chi0)
    assert_parity(gpu_maps(ctx, d), write_grid(d), label=f"lsa {psi0}/{chi0}")


@pytest.mark.parametrize("schedule", [capi.HAMX_SCHED_AUTO, capi.HAMX_SCHED_WAVE,
                                      capi.HAMX_SCHED_THREAD])
@pytest.mark.parametrize("nside_out", [32, 8])
def test_nan_on_a_large_shell_is_an_error(ctx, schedule, nside_out):
    """The same on a shell whose march leaves the check to a scan of the shell
    maps, written to the output or interpolated (which skips a NaN): one
    vertex, far enough out that few of the 12288 rays meet its cells."""
    print("case: nan on a large shell", schedule, nside_out, flush=True)
    par = Param(text=configs.random_forward(shell_num=1, nside_sim=32, nside_out=nside_out,
                                            oc_r_res=0.2, grid=(32, 32, 16)))
    d = par.los_desc(schedule=schedule)
    b, te, box = random_grids((32, 32, 16), seed=22)
    bad = tuple(a.copy() for a in b)
    bad[2][(26 * 32 + 10) * 16 + 5] = np.nan
    kw = dict(brnd_box=box, ternd=te, ternd_box=box)
    with pytest.raises(HamxError) as e:
        gpu_maps(ctx, d, brnd=bad, **kw)
    assert e.value.code == capi.HAMX_ERR_ARG and "non-finite" in str(e.value)
    assert_parity(gpu_maps(ctx, d, brnd=b, **kw), write_grid(d, brnd=b, **kw), label="after-nan")
