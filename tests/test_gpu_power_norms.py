"""Norms at the sizes where their launches change (needs an MI355X): nodes on
both sides of one block, of the partial sums added on the host and of the most
blocks, against numpy in FP64 (compensated device sums: 1e-13).
"""
import numpy as np
import pytest

from test_gpu_fd_kernels import R, torch  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", ["f64", "f32"])
@pytest.mark.parametrize("law,nq,n", [
    ("euler", 2, [8, 8]), ("euler", 2, [13, 5]), ("euler", 4, [32, 64]), ("euler", 4, [34, 61]),
    ("euler", 4, [128, 64]), ("euler", 5, [73, 72]), ("advection", 4, [128, 64]),
    ("advection", 4, [131, 63]), ("advection", 8, [128, 129])])
def test_norms(torch, R, law, nq, n, dtype):
    print(f"norms {law} nq={nq} {n} {dtype}", flush=True)
    gm = R.GridManager(R.LobattoCell(nq, nq), R.brick([np.arange(k + 1) * 0.5 for k in n], (True,) * 2))
    dg = R.DGSEM.brick(gm, R.EulerLaw(2) if law == "euler" else R.AdvectionLaw(2), dtype=dtype)
    rng = np.random.default_rng(nq)
    q = torch.from_numpy(rng.standard_normal((dg.K, dg.ns, dg.Np))).to(dg.torch_dtype).cuda()
    x = q.double().cpu().numpy().astype(np.longdouble)
    w = np.asarray(gm.cell.weights_1d, dtype=np.longdouble)
    MJ = np.outer(w, w).reshape(-1)[None, :] / 16  # cells of 1/2 x 1/2
    for p in (1, 2, 3, 2.5):
        want = np.sum(MJ[:, None] * np.abs(x) ** p, axis=(0, 2)) ** (1 / np.longdouble(p))
        got = R.weightednorm(dg, q, p, componentwise=True)
        assert np.max(np.abs(got / want - 1)) <= 1e-13
    want = np.sum(MJ[:, None] * x, axis=(0, 2))
    scale = np.sum(MJ[:, None] * np.abs(x), axis=(0, 2))
    assert np.max(np.abs(dg.integrals(q) - want) / scale) <= 1e-13
