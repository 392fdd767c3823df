"""Right-hand sides of FP64 advection in weak form on warped 2-D cells of Nq = 8
(needs an MI355X): two nodes per lane beyond 20000 cells, with an odd number of
cells, whose last group has one cell of its two, and one node up to there.
Against the oracle at 1e-12, as the other FP64 right-hand sides; dq overwritten
and added to, all directions and the sum of each alone.
"""
import numpy as np
import pytest

import oracle as O
import problems as PB
from test_gpu_fd_curved_advection import warp2
from test_gpu_fd_kernels import R, rel_l2, torch  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,face", [([160, 125], "rusanov"), ([143, 141], "rusanov"),
                                    ([143, 141], "central")])
def test_rhs(torch, R, n, face):
    print(f"curved advection right-hand side {n} {face}", flush=True)
    nq, u = 8, [1.0, -0.6]
    coords = [PB.julia_range(-1, 1, k + 1) for k in n]
    grid = R.generate(R.GridManager(R.LobattoCell(nq, nq), R.brick(coords, (False, True))), warp=warp2)
    og = O.BrickGrid(nq, coords, (False, True), warp=warp2)
    P = og.point_fields()
    rng = np.random.default_rng(8)
    q = PB.advection_wave(P, 2, 0.0) + 1e-2 * rng.standard_normal(P[:, 0, :].size)
    want = np.zeros(q.size)
    O.DG(og, "advection", u=u, surface_flux=face).rhs(want, q.copy(), 0.0, increment=False)
    d0 = np.abs(want).max() * rng.uniform(-1, 1, q.size)
    total = 0.0
    for dirs in [None, [1], [2]]:
        dg = R.DGSEM(law=R.AdvectionLaw(2, u), grid=grid, dtype="f64", directions=dirs,
                     surface_numericalflux=R.CentralFlux() if face == "central" else R.RusanovFlux())
        dev = lambda x: torch.from_numpy(x.copy()).cuda().reshape(dg.K, 1, dg.Np).contiguous()  # noqa: E731
        for add in (False, True):
            qd, dq = dev(q), dev(d0)
            dg(dq, qd, 0.0, increment=add)
            dg.synchronize()
            got = dq.cpu().numpy().reshape(-1)
            if dirs is None:
                err = rel_l2(got, want + d0 if add else want)
                print(f"   add={add} {err:.2e}", flush=True)
                assert err <= 1e-12
            elif not add:
                total = total + got
    assert rel_l2(total, want) <= 1e-12
