"""Grids that are thin across x and y (GPU): every way of taking the grid against
the C oracle, ensembles of such boxes against single contexts, and the time of a
step against the same number of cells along x.

Tolerance 1e-12 relative per physical quantity, as in test_gpu_parity.py.  The
times: a row of cells along z needs two lanes a cell at most (its faces across x
are extra positions where rows are not packed whole), a sixth wave of y faces
and shorter marches; three times the time of the row along x is allowed for."""
import os

import numpy as np
import pytest

from hermeshd_amd.config import HDConfig
from test_gpu_parity import TOL, field_rel_err, smooth_state
from test_gpu_stage_launch import CASES, MIXED, PERIODIC

pytestmark = pytest.mark.gpu

# one cell across; rows of three cells (a tile ends short of 64); eight and nine
# (whole rows of periodic grids, rows with an extra position); planes of a few
# cells, whose tiles span several segments
SIZES = [(1, 1, 200), (1, 70, 9), (2, 3, 50), (3, 1, 77), (8, 2, 31), (9, 2, 31)]


def solver_with(cfg, planes):
    from hermeshd_amd.solver import Solver
    old = os.environ.get("HD_STAGE_PLANES")
    if planes is not None:
        os.environ["HD_STAGE_PLANES"] = planes
    try:
        return Solver(cfg)
    finally:
        if planes is not None:
            os.environ.pop("HD_STAGE_PLANES") if old is None else os.environ.update(HD_STAGE_PLANES=old)


@pytest.mark.parametrize("bc", [PERIODIC, MIXED], ids=["periodic", "mixed"])
@pytest.mark.parametrize("name", list(CASES))
def test_thin_grids_match_oracle(oracle_mod, name, bc):
    import torch
    for n in SIZES:
        cfg = HDConfig(nx=n[0], ny=n[1], nz=n[2], lx=0.1 * n[0], ly=0.1 * n[1], lz=0.1 * n[2], bc=bc, T_floor=1e-4,
                       limiter=True, **CASES[name])
        q0 = smooth_state(cfg, seed=3)
        o = oracle_mod.Oracle(cfg.as_ints())
        ref, r1, r2 = q0.copy(), np.zeros_like(q0), np.zeros_like(q0)
        t, dt = np.array(0.0), np.array(0.0)
        o.step(ref, r1, r2, t, dt)
        for planes in (None, "-1", "0", "1", "4"):
            print(f"[thin] {name} {n} planes {planes}", flush=True)
            s = solver_with(cfg, planes)
            q = torch.from_numpy(q0.copy()).cuda()
            s.step(q, torch.zeros_like(q))
            s.check()
            assert field_rel_err(q.cpu().numpy(), ref) < TOL, (n, planes)


@pytest.mark.parametrize("choice", [0, 2, 7, 12])
def test_ensemble_of_thin_boxes_equals_single(choice):
    """Bitwise each context's own right-hand side, noise included."""
    import torch
    from hermeshd_amd.ensemble import Ensemble
    from hermeshd_amd.solver import Solver
    dims = [(1, 1, 130), (4, 4, 33), (9, 1, 40), (2, 31, 5)]
    base = HDConfig(nx=1, ny=1, nz=130, lx=1., ly=1., lz=130., nbasis=4, iquad=2, nQ=11, ivis=0, coll=3.0, colvis=0.5,
                    riemann="hllc", integrator="heun", noise=True, eta_sd=0.02, seed=5, realization=3, T_floor=1e-4)
    ens = Ensemble(base, dims)
    ens.set_launch(choice)
    cfgs = [base.replace(nx=d[0], ny=d[1], nz=d[2], lx=1. * d[0], ly=1. * d[1], lz=1. * d[2],
                         realization=base.realization + r) for r, d in enumerate(dims)]
    qs = [smooth_state(c, seed=9 + r) for r, c in enumerate(cfgs)]
    out = ens.views(ens.rhs(ens.pack(qs)))
    for r, c in enumerate(cfgs):
        assert torch.equal(Solver(c).rhs(torch.from_numpy(qs[r]).cuda()), out[r]), f"box {r}"


def step_time(cfg, dt=1e-5):
    import torch
    from hermeshd_amd.solver import Solver
    s, q = Solver(cfg), torch.from_numpy(smooth_state(cfg, seed=3)).cuda()
    q1, q2, d = torch.zeros_like(q), torch.zeros_like(q), torch.tensor(dt, dtype=torch.float64, device="cuda")
    best = 1e9
    for _ in range(4):
        a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        a.record()
        for _ in range(5):
            s.update(q, q1, q2, d)
        b.record()
        b.synchronize()
        best = min(best, a.elapsed_time(b) / 5)
    return best


@pytest.mark.parametrize("name", ["nb4", "nb10", "nb10_13"])
@pytest.mark.parametrize("n", [(1, 1, 65536), (2, 2, 16384), (4, 4, 4096), (1, 256, 256)],
                         ids=lambda d: "x".join(map(str, d)))
@pytest.mark.parametrize("bc", [PERIODIC, ("outflow", "outflow") + PERIODIC[2:]], ids=["periodic", "open"])
def test_thin_grids_keep_their_lanes(name, n, bc):
    mk = lambda d: HDConfig(nx=d[0], ny=d[1], nz=d[2], lx=0.1 * d[0], ly=0.1 * d[1], lz=0.1 * d[2], bc=bc,
                            T_floor=1e-4, limiter=False, **CASES[name])
    thin, row = step_time(mk(n)), step_time(mk((n[0] * n[1] * n[2], 1, 1)))
    print(f"[thin] {name} {n}: {thin * 1e3:.0f} us, along x {row * 1e3:.0f} us", flush=True)
    assert thin < 3 * row
