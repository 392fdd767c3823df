"""Right-hand sides of FP32 advection on 1-D grids large enough for a lane per
cell (needs an MI355X): both geometries, boundaries, remainders in the last wave
and dq accumulated into, against the oracle at the FP32 bar of
test_gpu_parity.py (1e-4).
"""
import numpy as np
import pytest

import oracle as O
import problems as PB
from test_gpu_fd_kernels import R, rel_l2, torch  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("geometry", ["auto", "general"])
@pytest.mark.parametrize("flux", ["rusanov", "central"])
@pytest.mark.parametrize("nq", range(2, 9))
def test_rhs(torch, R, nq, flux, geometry):
    K = 400000 // nq + (1 if nq % 2 else 63)  # just above the switch
    print(f"1-D cells nq={nq} K={K} {flux} {geometry}", flush=True)
    coords, per = [np.arange(K + 1) * 1.0], (nq % 2 == 0,)
    grid = R.generate(R.GridManager(R.LobattoCell(nq), R.brick(coords, per)))
    dg = R.DGSEM(law=R.AdvectionLaw(1, [-0.7]), grid=grid, dtype="f32", geometry=geometry,
                 surface_numericalflux=R.RusanovFlux() if flux == "rusanov" else R.CentralFlux())
    odg = O.DG(O.BrickGrid(nq, coords, per), "advection", u=[-0.7], surface_flux=flux)
    rng = np.random.default_rng(nq)
    qd = torch.from_numpy(rng.standard_normal((K, 1, nq))).float().cuda()
    qh = qd.double().cpu().numpy().reshape(-1)
    L = np.zeros(qh.size)
    odg.rhs(L, qh.copy(), 0.0, increment=False)
    for increment in (False, True):
        dq = torch.from_numpy(rng.standard_normal((K, 1, nq))).float().cuda()
        want = L + dq.double().cpu().numpy().reshape(-1) if increment else L
        dg(dq, qd, 0.0, increment=increment)
        dg.synchronize()
        err = rel_l2(dq.double().cpu().numpy().reshape(-1), want)
        print(f"   {increment}: {err:.2e}", flush=True)
        assert err <= 1e-4
