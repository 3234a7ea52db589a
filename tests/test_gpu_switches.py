"""The switches that select a cross-check kernel (GPU): that they do, and that
the kernels they select are right."""
import numpy as np
import pytest
import torch

import test_gpu_adjoint as adjoint
from hermeshd_amd import ics
from hermeshd_amd.config import HDConfig
from test_gpu_parity import CASES, TOL, field_rel_err, smooth_state

pytestmark = pytest.mark.gpu


def solver(cfg, monkeypatch, **env):
    from hermeshd_amd.solver import Solver
    with monkeypatch.context() as m:
        for k, v in env.items():
            m.setenv(k, v)
        return Solver(cfg)


# ------------------------------------------------- table-driven 13 moments ---
@pytest.mark.parametrize("env", [{"HD_FACES": "table"}, {"HD_KERNELS": "generic", "HD_LIMITER": "table"}],
                         ids=["faces", "generic"])
@pytest.mark.parametrize("name", ["tm13_nb4_roe_periodic", "tm13_nb10_roe_walls", "tm13_nb10_hllc_ivis0_outflow",
                                  "tgv_nb10_roe_8"])
def test_table_driven_13_moments(oracle_mod, monkeypatch, name, env):
    """HD_FACES=table runs the 13-moment model on k_face_flux and k_cell13: the
    context then holds the face fluxes, which the fused stage does not need."""
    cfg = CASES[name]
    q = ics.taylor_green(cfg) if name.startswith("tgv") else smooth_state(cfg, seed=5)
    s, plain = solver(cfg, monkeypatch, **env), solver(cfg, monkeypatch)
    nx, ny, nz = cfg.nx, cfg.ny, cfg.nz
    faces = (nx + 1) * ny * nz + nx * (ny + 1) * nz + nx * ny * (nz + 1)
    assert s.device_bytes - plain.device_bytes == 8 * cfg.iquad ** 2 * 13 * faces
    o = oracle_mod.Oracle(cfg.as_ints())
    qd = torch.from_numpy(q.copy()).cuda()
    q1d = torch.zeros_like(qd)
    q1, q2 = np.zeros_like(q), np.zeros_like(q)
    t, dt = np.array(0.0), np.array(0.0)
    for _ in range(3):
        o.step(q, q1, q2, t, dt)
        s.step(qd, q1d)
    s.check()
    assert field_rel_err(qd.cpu().numpy(), q) < TOL


# ----------------------------------------------------- per-cell transposes ---
def _two_point(names):
    return [n for n in names if adjoint.CFGS[n].nbasis != 10]


@pytest.mark.parametrize("name", _two_point(adjoint.CFGS))
def test_per_cell_rhs_vjp(oracle_mod, monkeypatch, name):
    monkeypatch.setenv("HD_VJP", "fused")
    adjoint.test_rhs_vjp_matches_autograd(torch.device("cuda:0"), oracle_mod, name)


@pytest.mark.parametrize("name,stage", [("nb4_nq11_hllc_noslip_ivis1", 2), ("nb4_nq11_hllc_walls_ivis0", 1),
                                        ("nb4_nq11_hllc_inflow_ivis1", 3), ("nb8_nq5_central_outflow", 2),
                                        ("nb4_nq11_roe_walls_ivis1", 2), ("nb4_nq13_roe_periodic_ivis1", 3)])
def test_per_cell_stage_vjp(oracle_mod, monkeypatch, name, stage):
    monkeypatch.setenv("HD_VJP", "fused")
    adjoint.test_stage_vjp_matches_autograd(torch.device("cuda:0"), oracle_mod, name, stage)


@pytest.mark.parametrize("nb,nq", [(4, 5), (4, 11), (8, 5), (8, 11), (4, 13), (10, 5), (10, 13)])
def test_fused_selects_another_transpose(monkeypatch, nb, nq):
    """The per-cell kernel sums in another order than the default of a small
    grid: equal to rounding, in some of the values not bitwise."""
    extra = dict(coll_q=2.0, col_q=0.3) if nq == 13 else {}
    visc = dict(ivis=1, coll=3.0, colvis=0.2) if nq >= 11 else {}
    cfg = HDConfig(nx=9, ny=7, nz=5, lx=0.9, ly=0.7, lz=0.5, nbasis=nb, iquad=3 if nb == 10 else 2, nQ=nq,
                   riemann="hllc", bc=("periodic",) * 6, T_floor=1e-4, limiter=False, integrator="heun", **visc,
                   **extra)
    q = torch.from_numpy(smooth_state(cfg, seed=4)).cuda()
    lam = torch.from_numpy(np.random.default_rng(3).standard_normal(q.shape)).cuda()
    a = solver(cfg, monkeypatch).rhs_vjp(q, lam)
    b = solver(cfg, monkeypatch, HD_VJP="fused").rhs_vjp(q, lam)
    assert field_rel_err(a.cpu().numpy(), b.cpu().numpy()) < adjoint.VJP_TOL
    assert not torch.equal(a, b)


# ------------------------------------------------ ways of taking the stage ---
@pytest.mark.parametrize("name", ["vortex_nb10_rows64", "relax_nq11_rows64", "vortex_nb10_hllc", "relax_nq11_bodyforce",
                                  "tm13_nb10_rows64"])
def test_stage_forms_agree(monkeypatch, name):
    """Equal runs of planes and items of one and of three planes run the same
    kernel on the same lanes: bitwise the same steps.  Five waves a tile are
    another kernel, whose contractions may differ: to rounding."""
    cfg = CASES[name]
    q0 = torch.from_numpy(smooth_state(cfg, seed=8)).cuda()
    outs = {}
    for planes in ("-1", "0", "1", "3"):
        s, q = solver(cfg, monkeypatch, HD_STAGE_PLANES=planes), q0.clone()
        q1 = torch.zeros_like(q)
        for _ in range(3):
            s.step(q, q1)
        s.check()
        outs[planes] = q
    assert torch.equal(outs["0"], outs["1"]) and torch.equal(outs["0"], outs["3"])
    assert field_rel_err(outs["-1"].cpu().numpy(), outs["0"].cpu().numpy()) < 1e-13
