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


@pytest.mark.parametrize("dtype", ["f64", "f32"])
@pytest.mark.parametrize("nq", range(2, 9))
def test_2d_small_advection_in_a_batch(torch, R, nq, dtype):
    """One node per lane (the operator alone on a small grid) and four (the
    batch's kernels, a work list and a launch of the kind's own) give the same
    bits: random states, a and b_dt away from zero."""
    rng = np.random.default_rng(nq)
    dgs, states = [], []
    for n in ([3, 2], [40, 41]):
        gm = R.GridManager(R.LobattoCell(nq, nq),
                           R.brick([PB.julia_range(-1, 1, k + 1) for k in n], (True, False)))
        dg = R.DGSEM(law=R.AdvectionLaw(2, [1.0, 0.7]), grid=R.generate(gm), dtype=dtype)
        dgs.append(dg)
        states.append([torch.from_numpy(rng.standard_normal((dg.K, dg.ns, dg.Np)))
                       .to(dg.torch_dtype).cuda() for _ in range(2)])
    want = []
    for dg, (q, d) in zip(dgs, states):
        qo, dq = torch.empty_like(q), d.clone()
        dg.lsrk_stage(qo, q, dq, -0.7, 3e-3)
        want.append((qo, dq))
    batch = R.Batch(dgs)
    for items in (1, 1 << 30):  # every kind on its own; all in the work list
        batch.configure(own_launch_items=items)
        qo, dq = [torch.empty_like(q) for q, _ in states], [d.clone() for _, d in states]
        batch.stage(qo, [q for q, _ in states], dq, [-0.7] * 2, [3e-3] * 2)
        torch.cuda.synchronize()
        for k in range(2):
            assert torch.equal(qo[k], want[k][0]) and torch.equal(dq[k], want[k][1])
    batch.close()
