"""Advection in flux-differencing form on warped cells (needs an MI355X): the
node kernel takes each node's u . l_d from LDS.  Against the oracle at the bars
of test_gpu_fluxdiff.py (FP64 1e-12, FP32 1e-4), all directions and each alone,
with cells that leave remainders in the workgroups.
"""
import numpy as np
import pytest

import oracle as O
import problems as PB
from test_gpu_fd_kernels import R, rel_l2, torch  # noqa: F401

pytestmark = pytest.mark.gpu


def warp2(x, y):
    return x + 0.05 * np.sin(np.pi * y), y + 0.05 * np.sin(np.pi * x)


def warp3(x, y, z):
    return (x + 0.05 * np.sin(np.pi * y), y + 0.05 * np.sin(np.pi * z),
            z + 0.05 * np.sin(np.pi * x))


@pytest.mark.parametrize("dtype", ["f64", "f32"])
@pytest.mark.parametrize("dim,nq,n,face", [
    (2, 2, [17, 9], "central"), (2, 5, [7, 5], "rusanov"), (2, 8, [3, 5], "central"),
    (3, 3, [5, 3, 4], "rusanov"), (3, 4, [2, 3, 3], "central"), (3, 6, [1, 2, 2], "rusanov"),
    (3, 8, [2, 1, 2], "central")])
def test_warped_stage(torch, R, dim, nq, n, face, dtype):
    print(f"fd curved advection dim={dim} nq={nq} {n} {face} {dtype}", flush=True)
    coords = [PB.julia_range(-1, 1, k + 1) for k in n]
    per, warp = (False,) * dim, warp2 if dim == 2 else warp3
    u = [1.0, -0.6, 0.3][:dim]
    grid = R.generate(R.GridManager(R.LobattoCell(*([nq] * dim)), R.brick(coords, per)), warp=warp)
    og = O.BrickGrid(nq, coords, per, warp=warp)
    odg = O.DG(og, "advection", u=u, volume_flux="central", surface_flux=face)
    P = og.point_fields()
    q = PB.advection_wave(P, dim, 0.0) + 1e-2 * np.random.default_rng(3).standard_normal(P[:, 0, :].size)
    total = 0.0
    for dirs in [None] + [[d + 1] for d in range(dim)]:
        dg = R.DGSEM(law=R.AdvectionLaw(dim, u), grid=grid, dtype=dtype, directions=dirs,
                     surface_numericalflux=R.CentralFlux() if face == "central" else R.RusanovFlux(),
                     volume_form=R.FluxDifferencingForm(R.CentralFlux()))
        qd = torch.from_numpy(q).to(dg.torch_dtype).cuda().reshape(dg.K, 1, dg.Np).contiguous()
        dq = dg.GridArray(0.0)
        dg(dq, qd, 0.0, increment=False)
        dg.synchronize()
        got = dq.double().cpu().numpy().reshape(-1)
        if dirs is None:
            want = np.zeros(q.size)
            odg.rhs(want, qd.double().cpu().numpy().reshape(-1).copy(), 0.0, increment=False)
            err = rel_l2(got, want)
            print(f"   dq {err:.2e}", flush=True)
            assert err <= (1e-12 if dtype == "f64" else 1e-4)
        else:
            total = total + got
    assert rel_l2(total, want) <= (1e-12 if dtype == "f64" else 1e-4)
