"""GatherScatter for every number of fields, and the reductions over the states
at node counts around their strides (needs an MI355X).

gather!'s fold is bit-exact (ascending rows, from zero); the reductions are
compensated sums, within 1e-14 of the sum of magnitudes (a few roundings).
"""
import numpy as np
import pytest

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


def make(R, dim, nq, n, law, dtype):
    coords = [PB.julia_range(0, 1, k + 1) for k in n]
    per = (True, False, True)[:dim] if n[0] > 1 else (False,) * dim
    grid = R.generate(R.GridManager(R.LobattoCell(*([nq] * dim)), R.brick(coords, per)))
    lawobj = R.AdvectionLaw(dim) if law == "advection" else R.EulerLaw(dim)
    return grid, R.DGSEM(law=lawobj, grid=grid, dtype=dtype)


@pytest.mark.parametrize("dtype", ["f64", "f32"])
@pytest.mark.parametrize("dim,nq,n", [(1, 5, [7]), (2, 4, [5, 3]), (3, 3, [4, 3, 5])])
@pytest.mark.parametrize("nf", [1, 2, 3, 4, 5, 7])
def test_gather_scatter_fields(torch, R, dim, nq, n, nf, dtype):
    grid, dg = make(R, dim, nq, n, "advection", dtype)
    rng = np.random.default_rng(nf)
    npt = np.float64 if dtype == "f64" else np.float32
    x = rng.standard_normal((dg.K, nf, dg.Np)).astype(npt)
    want = np.zeros((nf, grid.ncontinuous), dtype=npt)
    at = grid.dtoc.reshape(-1) - 1
    flat = x.transpose(1, 0, 2).reshape(nf, -1)
    for i in range(at.size):  # ascending rows
        want[:, at[i]] += flat[:, i]
    src = torch.from_numpy(x).cuda()
    c = torch.full((nf, grid.ncontinuous), 3.0, dtype=src.dtype, device="cuda")
    d = torch.empty_like(src)
    dg.gather(c, src, nf)
    dg.scatter(d, c, nf)
    dg.synchronize()
    assert np.array_equal(c.cpu().numpy(), want)
    assert np.array_equal(d.cpu().numpy().transpose(1, 0, 2).reshape(nf, -1), want[:, at])


@pytest.mark.parametrize("dtype", ["f64", "f32"])
@pytest.mark.parametrize("dim,nq,n,law", [
    (1, 2, [1], "euler"), (1, 5, [40], "advection"), (1, 8, [9000], "euler"),
    (2, 2, [130, 127], "euler"), (2, 7, [9, 31], "advection"), (2, 8, [60, 70], "euler"),
    (3, 6, [5, 3, 2], "euler"), (3, 8, [11, 10, 12], "euler"), (3, 7, [9, 8, 7], "advection")])
def test_reductions(torch, R, dim, nq, n, law, dtype):
    grid, dg = make(R, dim, nq, n, law, dtype)
    rng = np.random.default_rng(7)
    q = rng.standard_normal((dg.K, dg.ns, dg.Np)) + np.arange(dg.ns)[None, :, None]
    qd = torch.from_numpy(q).to(dg.torch_dtype).cuda().contiguous()
    h = qd.double().cpu().numpy().astype(np.longdouble)
    MJ = grid.MJ.astype(np.longdouble)[:, None, :]
    for got, f, root in ((dg.integrals(qd), lambda v: v, 1),
                         (R.weightednorm(dg, qd, componentwise=True), lambda v: v * v, 2),
                         (R.weightednorm(dg, qd, 3, componentwise=True), lambda v: np.abs(v) ** 3, 3)):
        want = (MJ * f(h)).sum(axis=(0, 2))
        scale = (MJ * np.abs(f(h))).sum(axis=(0, 2))
        assert np.all(np.abs(np.asarray(got, np.longdouble) ** root - want) <= 1e-14 * scale)
    top = R.weightednorm(dg, qd, float("inf"), componentwise=True)
    assert np.array_equal(top, np.abs(h).max(axis=(0, 2)).astype(np.float64))
    qd[dg.K // 2, dg.ns - 1, 1] = float("nan")
    assert np.isnan(R.weightednorm(dg, qd, float("inf"), componentwise=True)[-1])
    assert np.isnan(dg.integrals(qd)[-1])
