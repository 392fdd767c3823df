"""The 3-D column kernel packed across waves and with a wave per cell (needs an
MI355X): the same operations per cell, so any split of the launch gives the
same bits.  Cell counts on both sides of the switches (1024 cells of Nq = 6,
2048 of Nq = 7, operators beyond 256 MB), with remainders, against the oracle at
the bars of test_gpu_parity.py (FP64 1e-12; FP32 right-hand sides 1e-4, q_out
1e-6), and a relaxation step, whose product slots follow the launch.
"""
import ctypes

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


def make(R, nq, n, dtype, geometry):
    coords = [PB.julia_range(0, 10, k + 1) for k in n]
    per = (True, True, False)
    grid = R.generate(R.GridManager(R.LobattoCell(nq, nq, nq), R.brick(coords, per)))
    dg = R.DGSEM(law=R.EulerLaw(3), grid=grid, dtype=dtype, geometry=geometry)
    og = O.BrickGrid(nq, coords, per)
    P = og.point_fields()
    rng = np.random.default_rng(2)
    q = PB.isentropic_vortex_3d(P, 0.0, centre=(5.0, 5.0),
                                noise=1e-2 * rng.uniform(-1, 1, P[:, 0, :].shape))
    return dg, O.DG(og, "euler"), q


@pytest.mark.parametrize("dtype", ["f64", "f32"])
@pytest.mark.parametrize("geometry", ["auto", "general"])
@pytest.mark.parametrize("nq,n", [(5, [3, 2, 1]), (5, [13, 9, 11]), (6, [1, 1, 1]), (6, [11, 9, 10]),
                                  (6, [11, 11, 9]), (7, [2, 1, 3]), (7, [13, 12, 13]),
                                  (7, [13, 13, 13])])
def test_stage_on_both_sides(torch, R, nq, n, geometry, dtype):
    print(f"plane3 packing nq={nq} {n} {geometry} {dtype}", flush=True)
    if n == [1, 1, 1]:
        n = [1, 1, 2]
    dg, odg, q = make(R, nq, n, dtype, geometry)
    qd = torch.from_numpy(q).to(dg.torch_dtype).cuda().reshape(dg.K, dg.ns, dg.Np).contiguous()
    qh = qd.double().cpu().numpy().reshape(-1).copy()
    L = np.zeros(q.size)
    odg.rhs(L, qh, 0.0, increment=False)
    dq0 = 0.1 * np.abs(L).max() * np.random.default_rng(6).uniform(-1, 1, q.size)
    dqd = torch.from_numpy(dq0).to(dg.torch_dtype).cuda().reshape(qd.shape).contiguous()
    want = -0.6 * dqd.double().cpu().numpy().reshape(-1) + L
    qo = torch.empty_like(qd)
    dg.lsrk_stage(qo, qd, dqd, -0.6, 1e-4)
    dg.synchronize()
    e1 = rel_l2(dqd.double().cpu().numpy().reshape(-1), want)
    e2 = rel_l2(qo.double().cpu().numpy().reshape(-1), qh + 1e-4 * want)
    print(f"   dq {e1:.2e}, q_out {e2:.2e}", flush=True)
    assert e1 <= (1e-12 if dtype == "f64" else 1e-4)
    assert e2 <= (1e-12 if dtype == "f64" else 1e-6)


@pytest.mark.parametrize("dtype", ["f64", "f32"])
@pytest.mark.parametrize("nq,small,large", [(5, 12, 37), (6, 10, 31), (7, 12, 27)])
def test_small_and_large_launches_agree(torch, R, nq, small, large, dtype):
    """A state that repeats with the period of the small periodic brick's cells
    gives every copy of a cell the small brick's stage, bit for bit (the large
    brick lies beyond the Infinity Cache in FP64)."""
    def brick(k):
        gm = R.GridManager(R.LobattoCell(nq, nq, nq),
                           R.brick([np.arange(k + 1) * 1.0] * 3, (True,) * 3))
        return gm, R.DGSEM.brick(gm, R.EulerLaw(3), dtype=dtype)

    out = []
    rng = np.random.default_rng(1)
    one = np.stack([1 + 0.1 * rng.uniform(-1, 1, nq ** 3)]
                   + [0.1 * rng.uniform(-1, 1, nq ** 3) for _ in range(3)]
                   + [2.5 + 0.1 * rng.uniform(-1, 1, nq ** 3)])
    for k in (small, large):
        _, dg = brick(k)
        q = torch.from_numpy(one).to(dg.torch_dtype).cuda()[None].repeat(dg.K, 1, 1).contiguous()
        dq, qo = dg.GridArray(0.25), torch.empty_like(q)
        dg.lsrk_stage(qo, q, dq, -0.6, 1e-3)
        dg.synchronize()
        assert bool((dq == dq[:1]).all()) and bool((qo == qo[:1]).all())
        out.append((dq[0].clone(), qo[0].clone()))
    assert torch.equal(out[0][0], out[1][0]) and torch.equal(out[0][1], out[1][1])


@pytest.mark.parametrize("nq,n", [(5, [7, 5, 6]), (6, [10, 10, 11]), (7, [12, 13, 14])])
def test_relaxation_step(torch, R, nq, n):
    print(f"plane3 relaxation nq={nq} {n}", flush=True)
    dg, odg, q = make(R, nq, n, "f64", "auto")
    dt = 0.02 / max(n) / nq ** 2
    qd = torch.from_numpy(q).cuda().reshape(dg.K, dg.ns, dg.Np).contiguous()
    solver = R.RLSRK54(dg, qd, dt)
    R.dostep_(qd, solver)
    want, g = q.copy(), ctypes.c_double(1.0)
    z = [np.zeros(q.size) for _ in range(3)]
    O.lib().orc_dg_rlsrk_step(odg.h, 54, want, *z, 0.0, dt, ctypes.byref(g))
    got = qd.cpu().numpy().reshape(-1)
    print(f"   q {rel_l2(got, want):.2e}, gamma {solver.gamma!r} vs {g.value!r}", flush=True)
    assert rel_l2(got, want) <= 1e-12
