"""The fused stage's ways of taking a grid (five waves a tile, equal runs of
planes, items of n planes) at the edges of its 63-cell tiles, against the C
oracle (GPU).

Tolerance 1e-12 relative per physical quantity, as in test_gpu_parity.py: both
sides compute in FP64 and differ by contraction and summation order only."""
import os

import numpy as np
import pytest

from hermeshd_amd.config import HDConfig
from test_gpu_parity import TOL, field_rel_err, smooth_state

pytestmark = pytest.mark.gpu

PERIODIC = ("periodic",) * 6
MIXED = ("outflow", "outflow", "noslip", "wall", "periodic", "periodic")
CASES = {
    "nb4": dict(nbasis=4, iquad=2, nQ=5, riemann="hllc", integrator="heun"),
    "nb8": dict(nbasis=8, iquad=2, nQ=5, riemann="roe", integrator="heun"),
    "nb10": dict(nbasis=10, iquad=3, nQ=5, riemann="hllc", integrator="shu-osher"),
    "nb4_stress": dict(nbasis=4, iquad=2, nQ=11, ivis=1, coll=20.0, colvis=0.5, riemann="hllc", integrator="heun",
                       body_force=(0.02, -0.01, 0.03)),
    "nb4_noise": dict(nbasis=4, iquad=2, nQ=11, ivis=0, coll=3.0, colvis=0.5, riemann="hllc", integrator="heun",
                      noise=True, eta_sd=0.02),
    "nb10_stress": dict(nbasis=10, iquad=3, nQ=11, ivis=1, coll=30.0, colvis=0.4, riemann="central",
                        integrator="shu-osher"),
    "nb4_13": dict(nbasis=4, iquad=2, nQ=13, ivis=0, coll=3.0, colvis=0.2, coll_q=2.0, col_q=0.3, riemann="hllc",
                   integrator="heun"),
    "nb10_13": dict(nbasis=10, iquad=3, nQ=13, ivis=1, coll=30.0, colvis=0.4, coll_q=12.0, col_q=0.6, riemann="roe",
                    integrator="shu-osher"),
}
# one cell; a tile exactly, one short and one over; several tiles; planes that
# the items do not divide
SIZES = [(1, 1, 1), (62, 1, 3), (63, 2, 4), (64, 1, 5), (20, 13, 7)]


@pytest.fixture(scope="module")
def torch_mod():
    import torch
    assert torch.cuda.is_available(), "GPU tests need a ROCm device"
    return torch


@pytest.mark.parametrize("bc", [PERIODIC, MIXED], ids=["periodic", "mixed"])
@pytest.mark.parametrize("name", list(CASES))
def test_launch_forms_match_oracle(torch_mod, oracle_mod, name, bc):
    from hermeshd_amd.solver import Solver
    for n in SIZES:
        cfg = HDConfig(nx=n[0], ny=n[1], nz=n[2], lx=0.1 * n[0], ly=0.1 * n[1], lz=0.1 * n[2], bc=bc, T_floor=1e-4,
                       limiter=True, **CASES[name])
        q0 = smooth_state(cfg, seed=3)
        o = oracle_mod.Oracle(cfg.as_ints())
        ref, r1, r2 = q0.copy(), np.zeros_like(q0), np.zeros_like(q0)
        t, dt = np.array(0.0), np.array(0.0)
        o.step(ref, r1, r2, t, dt)
        for planes in ("-1", "0", "1", "3"):
            print(f"[stage_launch] {name} {n} planes {planes}", flush=True)
            old = os.environ.get("HD_STAGE_PLANES")
            os.environ["HD_STAGE_PLANES"] = planes
            try:
                s = Solver(cfg)
            finally:
                if old is None:
                    del os.environ["HD_STAGE_PLANES"]
                else:
                    os.environ["HD_STAGE_PLANES"] = old
            q = torch_mod.from_numpy(q0.copy()).cuda()
            s.step(q, torch_mod.zeros_like(q))
            s.check()
            assert field_rel_err(q.cpu().numpy(), ref) < TOL, (n, planes)


@pytest.mark.parametrize("dims", [[(1, 1, 1), (3, 1, 2)], [(23, 30, 29), (2, 3, 1), (31, 24, 27)]],
                         ids=["few_chunks", "runs_of_chunks"])
def test_ensemble_draw_equals_single(dims):
    """The ensemble's draw, fewer chunks than blocks and blocks that cross
    from one family or realization to the next: bitwise each context's own."""
    import torch
    from hermeshd_amd.ensemble import Ensemble
    from hermeshd_amd.solver import Solver
    nx, ny, nz = dims[0]
    base = HDConfig(nx=nx, ny=ny, nz=nz, lx=1. * nx, ly=1. * ny, lz=1. * nz, nbasis=4, iquad=2, nQ=11, ivis=0,
                    coll=3.0, colvis=0.5, riemann="hllc", integrator="heun", noise=True, eta_sd=0.02, seed=5,
                    realization=3, T_floor=1e-4)
    cfgs = [base.replace(nx=d[0], ny=d[1], nz=d[2], lx=1. * d[0], ly=1. * d[1], lz=1. * d[2],
                         realization=base.realization + r) for r, d in enumerate(dims)]
    ens = Ensemble(base, dims)
    qs = [smooth_state(c, seed=9 + r) for r, c in enumerate(cfgs)]
    out = ens.views(ens.rhs(ens.pack(qs)))
    for r, c in enumerate(cfgs):
        assert torch.equal(Solver(c).rhs(torch.from_numpy(qs[r]).cuda()), out[r]), f"realization {r}"


@pytest.mark.parametrize("dims", [(1, 1, 1), (2, 1, 3), (4, 4, 1), (7, 4, 1), (1, 29, 1), (8, 4, 2), (5, 3, 7)],
                         ids=lambda d: "x".join(map(str, d)))
@pytest.mark.parametrize("nb,riemann", [(4, "hllc"), (4, "central"), (10, "roe"), (10, "hllc")])
def test_periodic_13_moment_transpose_equals_per_cell(dims, nb, riemann):
    """The split 13-moment transpose at the edges of its tiles (28 or 64
    faces, 16 or 32 cells), directions of one cell included, against the
    per-cell kernel: every term of the stage map on, both with and without the
    limiter's state."""
    import torch
    from hermeshd_amd.solver import Solver
    nx, ny, nz = dims
    cfg = HDConfig(nx=nx, ny=ny, nz=nz, lx=1. * nx, ly=1. * ny, lz=1. * nz, nbasis=nb, iquad=3 if nb == 10 else 2,
                   nQ=13, ivis=1, coll=3.0, colvis=0.2, coll_q=2.0, col_q=0.3, riemann=riemann, bc=PERIODIC,
                   body_force=(0.02, -0.01, 0.03), limiter=True, T_floor=1e-4, integrator="heun")
    rng = np.random.default_rng(17)
    q = smooth_state(cfg, seed=2)
    dev = lambda a: torch.from_numpy(a).cuda()
    lam, acc, out, qn = (dev(rng.standard_normal(q.shape)) for _ in range(4))
    qd, res = dev(q), []
    for mode in ("split", "fused"):
        old = os.environ.get("HD_VJP")
        os.environ["HD_VJP"] = mode
        try:
            s = Solver(cfg)
        finally:
            os.environ.pop("HD_VJP") if old is None else os.environ.update(HD_VJP=old)
        for raw in (None, qd):
            lam_in = torch.empty_like(qd)
            dcoll = torch.zeros((), dtype=torch.float64, device="cuda")
            s.stage_vjp(qd, lam, lam_in, 1e-3, 0.25, 0.75, acc=[(1.0, acc), (0.5, qn)], q_raw=raw, out=out, qn=qn,
                        dcoll=dcoll)
            res.append((lam_in.cpu().numpy(), float(dcoll)))
        # with lam: in one cell the terms of a field may cancel to nothing
        res.append(((lam + s.rhs_vjp(qd, lam)).cpu().numpy(), 0.))
    for (a, da), (b, db) in zip(res[:3], res[3:]):
        assert field_rel_err(a, b) < TOL
        assert abs(da - db) <= TOL * max(abs(db), 1.0)


@pytest.mark.parametrize("dims", [(1, 1, 1), (15, 1, 1), (4, 4, 1), (5, 3, 7), (6, 4, 4)],
                         ids=lambda d: "x".join(map(str, d)))
@pytest.mark.parametrize("bc", [PERIODIC, MIXED, ("outflow",) * 2 + ("periodic",) * 2 + ("noslip", "outflow")],
                         ids=["periodic", "mixed", "outflow"])
@pytest.mark.parametrize("name", ["nb4", "nb8", "nb4_stress", "nb4_13"])
def test_transpose_of_a_point_a_lane(oracle_mod, name, bc, dims):
    """The two-point rules' transpose at the edges of its 16-cell tiles and at
    every kind of boundary, against automatic differentiation of the oracle's
    transcription, to the tolerance of test_gpu_adjoint.py (with lam added:
    in one cell the terms of a field may cancel to nothing)."""
    import torch
    from hermeshd_amd.solver import Solver
    from test_gpu_adjoint import DG, VJP_TOL
    nx, ny, nz = dims
    cfg = HDConfig(nx=nx, ny=ny, nz=nz, lx=1. * nx, ly=1. * ny, lz=1. * nz, bc=bc, T_floor=1e-4, limiter=False,
                   **CASES[name])
    q = smooth_state(cfg, seed=4)
    lam = np.random.default_rng(3).standard_normal(q.shape)
    dg = DG(cfg, oracle_mod.Oracle(cfg.as_ints()).tables())
    qt = torch.from_numpy(q).requires_grad_(True)
    (ref,) = torch.autograd.grad(dg.rhs(qt), qt, torch.from_numpy(lam))
    got = Solver(cfg).rhs_vjp(torch.from_numpy(q).cuda(), torch.from_numpy(lam).cuda()).cpu().numpy()
    assert field_rel_err(lam + got, lam + ref.numpy()) < VJP_TOL


@pytest.mark.parametrize("n", [(1, 1, 1), (255, 1, 1), (256, 2, 1), (27, 19, 1), (128, 16, 16), (331, 11, 9)],
                         ids=lambda d: "x".join(map(str, d)))
@pytest.mark.parametrize("name", ["nb4", "nb8", "nb10"])
@pytest.mark.parametrize("low", ["steep", "mean"])
def test_step_equals_min_dt_and_update(torch_mod, low, name, n):
    """One pass for the time step and the first limiter, in one block (two cells
    a thread), several, and in two passes again: bitwise min_dt and then
    update, with steep cells or cells of a mean below the floor, the last one
    (whose sound speed dt takes) among them."""
    from hermeshd_amd.solver import Solver
    cfg = HDConfig(nx=n[0], ny=n[1], nz=n[2], lx=0.1 * n[0], ly=0.1 * n[1], lz=0.1 * n[2], bc=PERIODIC, T_floor=1e-4,
                   rh_floor=0.05, limiter=True, **CASES[name])
    q = torch_mod.from_numpy(smooth_state(cfg, seed=6)).cuda()
    cells = q[1:, :5].flatten(2) if low == "steep" else q.flatten(2)
    cells[..., ::7] *= 12.0 if low == "steep" else 0.02
    cells[..., -1] *= 12.0 if low == "steep" else 0.02
    s, qa, qb = Solver(cfg), q.clone(), q.clone()
    t, dt = torch_mod.full_like(s.t, 0.25), torch_mod.zeros_like(s.dt)
    s.step(qa, torch_mod.zeros_like(q), t=t, dt=dt)
    ref = s.min_dt(qb)
    s.update(qb, torch_mod.zeros_like(q), None, ref)
    lim = q.clone()
    s.limit(lim)
    assert low == "steep" or not torch_mod.equal(lim, q)
    assert float(dt) == float(ref) and float(t) == 0.25 + float(ref)
    assert torch_mod.equal(qa, qb)
