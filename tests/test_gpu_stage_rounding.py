"""A stage rounds the state where its formula does, and nowhere else (GPU).

A stage's output is a*q_n + b*v with v = q + dt*R.  With R from hd_rhs and the
sum in extended precision (64 bits of mantissa), the output may be off by half a
unit in its last place (its own rounding), by b times that of v, by those of the
products a*q_n and b*v where they are not exact (a third and two thirds, and
three quarters), and by the rounding of the increment dt*R:
the terms of R are at most about 100 times R here (volume and faces cancel) and
some 50 roundings of 1.1e-16 enter it, so 1e-12 of the field's largest
increment is allowed for.  The increments are 1e-6 of the state and below, so
that this allowance is a hundredth of a unit in the last place of the means."""
import numpy as np
import pytest

from hermeshd_amd.config import HDConfig
from test_gpu_parity import smooth_state

pytestmark = pytest.mark.gpu

CASES = {
    "nb4": dict(nbasis=4, iquad=2, nQ=5, riemann="hllc", integrator="heun"),
    "nb8": dict(nbasis=8, iquad=2, nQ=5, riemann="roe", integrator="heun"),
    "nb10": dict(nbasis=10, iquad=3, nQ=5, riemann="hllc", integrator="shu-osher"),
    "nb4_stress": dict(nbasis=4, iquad=2, nQ=11, ivis=0, coll=2.0, colvis=0.5, riemann="hllc", integrator="heun"),
    "nb10_stress": dict(nbasis=10, iquad=3, nQ=11, ivis=0, coll=2.0, colvis=0.4, riemann="hllc",
                        integrator="shu-osher"),
    "nb10_13": dict(nbasis=10, iquad=3, nQ=13, ivis=0, coll=2.0, colvis=0.4, coll_q=2.0, col_q=0.3, riemann="roe",
                    integrator="shu-osher"),
}


@pytest.mark.parametrize("n", [(20, 13, 7), (70, 40, 33)], ids=["few_tiles", "runs"])
@pytest.mark.parametrize("name", list(CASES))
def test_roundings_at_the_state_size(name, n):
    import torch
    from hermeshd_amd.solver import Solver
    cfg = HDConfig(nx=n[0], ny=n[1], nz=n[2], lx=0.1 * n[0], ly=0.1 * n[1], lz=0.1 * n[2], bc=("periodic",) * 6,
                   T_floor=1e-4, limiter=False, **CASES[name])
    s, dev = Solver(cfg), lambda a: torch.from_numpy(a).cuda()
    q, qn = smooth_state(cfg, seed=3), smooth_state(cfg, seed=4)
    R = s.rhs(dev(q)).cpu().numpy()
    dt = 1e-6 / max(1.0, float(np.abs(R).max()))
    L = np.longdouble
    order = 3 if cfg.integrator == "shu-osher" else 2
    weights = {2: [(0.0, 1.0), (0.5, 0.5)], 3: [(0.0, 1.0), (0.75, 0.25), (1.0 / 3.0, 2.0 / 3.0)]}[order]
    for i, (a, b) in enumerate(weights):
        out = torch.empty_like(dev(q))
        s.stage(order, i + 1, dev(q), dev(qn), out, dt)
        got = out.cpu().numpy()
        ref = L(a) * qn.astype(L) + L(b) * (q.astype(L) + L(dt) * R.astype(L))
        err = np.abs(got.astype(L) - ref)
        slack = 1e-12 * dt * np.abs(R).max(axis=(0, 2, 3, 4))[None, :, None, None, None]
        half = 0.5 * np.spacing(np.abs(got))
        if a != 0.0:
            half = half + 0.5 * b * np.spacing(np.abs(q))
        if order == 3 and a != 0.0:
            half = half + 0.5 * np.spacing(a * np.abs(qn)) + (i == 2) * 0.5 * np.spacing(b * np.abs(q))
        bound = half + slack
        worst = float((err / bound)[0, [0, 4]].max())
        print(f"[rounding] {name} {n} stage {i + 1}: worst of rh, en {worst:.3f} of the bound", flush=True)
        assert (err <= bound * (1 + 1e-6)).all(), (i, float((err / bound).max()))


@pytest.mark.parametrize("nb", [4, 10])
def test_right_hand_side_reads_no_state_that_it_does_not_depend_on(nb):
    """With the stress relaxed implicitly its right-hand side is a function of
    the velocity alone: an infinite stress leaves it as it is."""
    import torch
    from hermeshd_amd.solver import Solver
    cfg = HDConfig(nx=9, ny=5, nz=4, lx=0.9, ly=0.5, lz=0.4, nbasis=nb, iquad=3 if nb == 10 else 2, nQ=11, ivis=1,
                   coll=2.0, colvis=0.5, riemann="central", bc=("periodic",) * 6, T_floor=1e-4, limiter=False,
                   integrator="heun")
    s, q = Solver(cfg), smooth_state(cfg, seed=3)
    ref = s.rhs(torch.from_numpy(q).cuda())
    q[0, 5, 2, 3, 4] = np.inf
    got = s.rhs(torch.from_numpy(q).cuda())
    assert torch.equal(got[:, 5:], ref[:, 5:])
