"""GPU checks of the grid-gradient scatter where the runs of samples within a
cell are longest and shortest: the FP64 sweeps merge the runs of 64
consecutive samples (8 at a time), the FP32 batch moves a lane's corner sums
from cell to cell.

Oracle: central differences of the GPU forward along a random direction, at
the step and with the bound of the other adjoint checks (truncation and
rounding both below 1e-7 of the derivative: rel 1e-6); the batches against
the plain adjoint at their stated 1e-9 (FP64) and 1e-4 (FP32).
"""
import numpy as np
import pytest

from hammurabix_amd import Param, _capi as capi, configs
from oracle_lib import rel_l2
from test_gpu_adjoint import adjoint, loss, random_grids, scaled_weights
from test_gpu_batch import (grids, instance, plain_adjoint_passes, scale_adjoint, with_adjoint)

pytestmark = pytest.mark.gpu

# grid, radial step [kpc]: one cell (a run is the chunk); a step longer than
# a cell (64 runs a chunk, more than the cell cache holds; cells passed
# over); runs of a few samples and partly filled rounds
CASES = [((2, 2, 2), 0.05), ((128, 128, 64), 0.8), ((17, 9, 33), 0.1)]


def desc(shape, res):
    return Param(text=configs.random_forward(nside_sim=4, nside_out=16, oc_r_res=res,
                                             grid=shape)).los_desc()


@pytest.mark.parametrize("shape,res", CASES)
def test_grid_gradient_of_long_and_short_runs(ctx, shape, res):
    print(f"case: adjoint runs {shape} {res}", flush=True)
    d = desc(shape, res)
    b, te, box = random_grids(shape, seed=31)
    te = np.ascontiguousarray(np.abs(te) + 1e-4)  # no sample at the te > 0 clamp
    g0 = dict(brnd=b, brnd_box=box, ternd=te, ternd_box=box)
    w = scaled_weights(ctx, d, g0, seed=32)
    _, g = adjoint(ctx, d, w, g0, with_grid=True)
    rng = np.random.default_rng(33)
    v = [rng.normal(size=a.shape) for a in b]
    vt = rng.normal(size=te.shape)
    for name, h, step in (
            ("brnd", 1e-5 * 2e-6, lambda s: dict(g0, brnd=tuple(
                np.ascontiguousarray(a + s * va) for a, va in zip(b, v)))),
            ("ternd", 1e-5 * 0.003, lambda s: dict(g0, ternd=np.ascontiguousarray(te + s * vt)))):
        fd = (loss(ctx, d, w, step(h)) - loss(ctx, d, w, step(-h))) / (2 * h)
        adj = (sum(float(np.dot(ga, va)) for ga, va in zip(g["dbrnd"], v)) if name == "brnd"
               else float(np.dot(g["dternd"], vt)))
        print(f"{name}: adjoint {adj:.10e} fd {fd:.10e}", flush=True)
        assert abs(adj - fd) <= 1e-6 * abs(fd)


@pytest.mark.parametrize("prec,tol", [(capi.HAMX_PREC_F64, 1e-9), (capi.HAMX_PREC_F32, 1e-4)])
@pytest.mark.parametrize("shape,res", CASES)
def test_batch_gradient_of_long_and_short_runs(ctx, shape, res, prec, tol):
    print(f"case: batch adjoint runs {shape} {res} precision {prec}", flush=True)
    sp = instance(4, 16, [1.4e9, 23e9], g=grids(shape, 34))
    sp["desc"] = desc(shape, res)
    specs = with_adjoint([sp], seed=35)
    with ctx.batch(specs, precision=prec, tune=False, adjoint=True) as bt:
        bt.run()
        scale_adjoint(specs)
        bt.run_adjoint()
        _, gb, gt = plain_adjoint_passes(ctx, sp)
        for name, a, r in zip(("bx", "by", "bz", "te"),
                              (*sp["grads"]["dbrnd"], sp["grads"]["dternd"]), (*gb, gt)):
            err = rel_l2(a.cpu().numpy(), r)
            print(f"d{name} rel L2 {err:.2e}", flush=True)
            assert err <= tol, name
