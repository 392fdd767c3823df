"""The weak-form stage kernels with a lane per node (needs an MI355X): 1-D
cells, and curved 2-D cells, whose FP32 handles read FP32 copies of the
geometry.  Every Nq, with cells that leave remainders in waves and workgroups,
boundaries, and both precisions, against the oracle at the bars of
test_gpu_parity.py (FP64 1e-12; FP32 right-hand sides 1e-4, q_out 1e-6).
"""
import numpy as np
import pytest

import oracle as O
import problems as PB

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def torch():
    import torch as t
    if not t.cuda.is_available():
        pytest.skip("no HIP device")
    return t


@pytest.fixture(scope="module")
def R(torch):
    import ravenhip
    return ravenhip


def rel_l2(a, b):
    return float(np.linalg.norm(a - b) / max(np.linalg.norm(b), 1e-300))


def check_stage(torch, R, dim, nq, n, law, dtype, geometry, warp=None):
    coords = [PB.julia_range(-1, 1, k + 1) for k in n]
    per = (True, False)[:dim] if n[0] > 1 else (False,) * dim
    gm = R.GridManager(R.LobattoCell(*([nq] * dim)), R.brick(coords, per))
    grid = R.generate(gm, warp=warp)
    u = [1.0, 0.5][:dim] if law == "advection" else None
    dg = R.DGSEM(law=R.AdvectionLaw(dim, u) if law == "advection" else R.EulerLaw(dim), grid=grid,
                 dtype=dtype, geometry=geometry)
    og = O.BrickGrid(nq, coords, per, warp=warp)
    odg = O.DG(og, law, u=u)
    P = og.point_fields()
    rng = np.random.default_rng(3)
    q = PB.advection_wave(P, dim, 0.0) if law == "advection" else PB.euler_wave(P, dim, 0.0)
    q = q + 1e-2 * rng.standard_normal(q.size)
    qd = torch.from_numpy(q).to(dg.torch_dtype).cuda().reshape(dg.K, dg.ns, dg.Np).contiguous()
    qh = qd.double().cpu().numpy().reshape(-1).copy()
    L = np.zeros(q.size)
    odg.rhs(L, qh, 0.0, increment=False)
    dqd = torch.from_numpy(0.1 * np.abs(L).max() * rng.uniform(-1, 1, q.size)).to(dg.torch_dtype)
    dqd = dqd.cuda().reshape(qd.shape).contiguous()
    want = -0.6 * dqd.double().cpu().numpy().reshape(-1) + L
    qo = torch.empty_like(qd)
    dg.lsrk_stage(qo, qd, dqd, -0.6, 1e-4)
    dg.synchronize()
    e1 = rel_l2(dqd.double().cpu().numpy().reshape(-1), want)
    e2 = rel_l2(qo.double().cpu().numpy().reshape(-1), qh + 1e-4 * want)
    print(f"   {dim}-D nq={nq} {n} {law} {dtype} {geometry}: dq {e1:.2e}, q_out {e2:.2e}", flush=True)
    assert e1 <= (1e-12 if dtype == "f64" else 1e-4)
    assert e2 <= (1e-12 if dtype == "f64" else 1e-6)


@pytest.mark.parametrize("dtype", ["f64", "f32"])
@pytest.mark.parametrize("law", ["euler", "advection"])
@pytest.mark.parametrize("geometry", ["auto", "general"])
@pytest.mark.parametrize("nq", range(2, 9))
def test_1d_stage(torch, R, nq, geometry, law, dtype):
    c = 64 // nq  # cells of a wave
    for K in (1, c, c + 1, 5 * c - 1):
        check_stage(torch, R, 1, nq, [K], law, dtype, geometry)


@pytest.mark.parametrize("dtype", ["f64", "f32"])
@pytest.mark.parametrize("law", ["euler", "advection"])
@pytest.mark.parametrize("nq", range(2, 9))
def test_2d_warped_stage(torch, R, nq, law, dtype):
    def warp(x, y):
        return x + 0.05 * np.sin(np.pi * y), y + 0.05 * np.sin(np.pi * x)

    for n in ([2, 1], [5, 3], [17, 7]):
        check_stage(torch, R, 2, nq, n, law, dtype, "auto", warp)


@pytest.mark.parametrize("law,dtype", [("advection", "f64"), ("advection", "f32"),
                                       ("euler", "f32")])
@pytest.mark.parametrize("nq", range(2, 9))
def test_2d_nodes_per_lane(torch, R, nq, law, dtype):
    """Affine 2-D cells that give a lane several nodes on large grids: both
    sides of the size where the launch changes over, and a remainder."""
    waves = {5: 2, 6: 4, 7: 4}.get(nq, 1)  # sharing a group's cells
    line = 64 * waves // nq**2 * (6144 // waves)
    for K in (line, line + 1, line + 37):
        check_stage(torch, R, 2, nq, [K, 1], law, dtype, "auto")
