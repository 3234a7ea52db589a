"""The switches that select a cross-check kernel (GPU): that they do, and that
the kernels they select are right."""
import os

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
