"""The ensemble's limiter over boxes of very different sizes (GPU): bitwise each
context's own, and on one large box no slower than twice a context's."""
import numpy as np
import pytest
import torch

from hermeshd_amd.config import HDConfig
from test_gpu_parity import smooth_state

pytestmark = pytest.mark.gpu


def base(n):
    return HDConfig(nx=n[0], ny=n[1], nz=n[2], lx=1. * n[0], ly=1. * n[1], lz=1. * n[2], nbasis=4, iquad=2, nQ=5,
                    riemann="hllc", integrator="heun", limiter=True, rh_floor=0.9, T_floor=0.5, bc=("periodic",) * 6)


def test_ensemble_limit_equals_single():
    from hermeshd_amd.ensemble import Ensemble
    from hermeshd_amd.solver import Solver
    dims = [(1, 1, 1), (70, 60, 50), (3, 1, 2), (16, 16, 16)]
    ens = Ensemble(base(dims[0]), dims)
    qs = [smooth_state(base(d), seed=r) for r, d in enumerate(dims)]
    q = ens.pack(qs)
    ens.limit(q)
    for d, s, got in zip(dims, qs, ens.views(q)):
        ref = torch.from_numpy(s).cuda()
        Solver(base(d)).limit(ref)
        assert torch.equal(got, ref), d
        assert d != (70, 60, 50) or not np.array_equal(ref.cpu().numpy(), s)


def test_one_large_box_fills_the_chip():
    from hermeshd_amd.ensemble import Ensemble
    from hermeshd_amd.solver import Solver
    cfg = base((160, 160, 160))
    ens, s = Ensemble(cfg, [(160, 160, 160)]), Solver(cfg)
    q = ens.zeros()
    v = ens.views(q)[0]
    v[0, 0], v[0, 4] = 1.0, 2.5

    def best(f):
        t = []
        for _ in range(5):
            a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            a.record()
            for _ in range(5):
                f()
            b.record()
            b.synchronize()
            t.append(a.elapsed_time(b) / 5)
        return min(t)

    te, ts = best(lambda: ens.limit(q)), best(lambda: s.limit(v))
    print(f"[ens_limit] ensemble {te * 1e3:.0f} us, context {ts * 1e3:.0f} us", flush=True)
    assert te < 2 * ts
