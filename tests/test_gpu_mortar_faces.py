"""mortar_face_kernel, a wave per sub-face (needs an MI355X): lists of
non-conforming faces that leave waves of a workgroup without a face, lists
with hanging or covered faces alone, and the smallest and largest Nq, against
the oracle's restatement at the bars of test_gpu_parity.py (FP64 1e-12, FP32
1e-4).  A face taken off the list is self-mapped, on both sides.
"""
import types

import numpy as np
import pytest

import oracle as O
import problems as PB
from test_gpu_parity import R, _adapted_grid, _ArrayGrid, _warp10, _warp10_2d, rel_l2, torch  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", ["f64", "f32"])
@pytest.mark.parametrize("dim,nq", [(2, 2), (2, 8), (3, 2), (3, 4), (3, 8)])
def test_face_lists(torch, R, dim, nq, dtype):  # noqa: F811
    grid = _adapted_grid(R, dim, nq, 4, 1, 2.5, _warp10 if dim == 3 else _warp10_2d)
    K, nfp, nsub = grid.K, nq ** (dim - 1), 2 ** (dim - 1)
    rng = np.random.default_rng(5)
    full = np.asarray(grid.face_kind).reshape(K, 2 * dim)
    hanging = np.argwhere(full == 1)
    assert len(hanging) % nsub == 0 and len(hanging) > nsub
    for keep_covered, nhang in ((True, len(hanging) - 1), (True, len(hanging) - nsub + 1),
                                (False, 1), (True, 0)):
        kind = np.where(full == 2, 2 if keep_covered else 0, 0).astype(np.int32)
        for e, f in hanging[rng.permutation(len(hanging))[:nhang]]:
            kind[e, f] = 1
        dg = R.DGSEM(law=R.EulerLaw(dim), grid=grid, dtype=dtype)
        dg.enable_mortars(types.SimpleNamespace(face_kind=kind,
                                                mortar_partner=grid.mortar_partner))
        ag = _ArrayGrid(grid)
        ag.points = grid.points
        surf = np.array(grid.surface).reshape(K, 2 * dim, nfp, dim + 2)
        surf_full = surf.reshape(-1).copy()
        surf[kind != 0, :, dim + 1] = 0.0
        ag.surf = surf.reshape(-1)
        odg = O.DG(ag, "euler")
        lower, upper = np.zeros(nq * nq), np.zeros(nq * nq)
        R._lib.check(R.lib().rv_lobatto_halves(nq, R._lib.ptr(lower, R._lib.ctypes.c_double),
                                               R._lib.ptr(upper, R._lib.ctypes.c_double)))
        vortex = PB.isentropic_vortex_3d if dim == 3 else PB.isentropic_vortex_2d
        q = vortex(grid.points, 0.0)
        q = q * (1 + 1e-3 * rng.uniform(-1, 1, q.size))
        qd = torch.from_numpy(q).to(dg.torch_dtype).cuda().reshape(K, dg.ns, dg.Np).contiguous()
        qh = qd.double().cpu().numpy().reshape(-1).copy()
        want = np.zeros(q.size)
        odg.rhs(want, qh.copy(), 0.0, increment=False)
        odg.mortar_add(kind.reshape(-1), grid.mortar_partner, lower, upper, surf_full, qh, want)
        got = dg.GridArray(0.0)
        dg(got, qd, 0.0, increment=False)
        dg.synchronize()
        err = rel_l2(got.double().cpu().numpy().reshape(-1), want)
        print(f"   {dim}-D nq={nq} {dtype}: {int((kind == 2).sum())} covered, {nhang} hanging: "
              f"{err:.2e}", flush=True)
        assert err <= (1e-12 if dtype == "f64" else 1e-4)
