"""Stages and right-hand sides beyond the 256 MB Infinity Cache (needs an
MI355X), where dq and q_out are streamed past the caches or cells change their
packing.  Every cell of a small periodic brick has a random state of its own; a
large brick of whole copies of it repeats the state, so each of its cells has the
small brick's result, from the oracle (FP64 1e-12; FP32 right-hand sides 1e-4,
q_out 1e-6).  A wrong neighbour, slab or remainder shows in any cell.  (Curved
3-D copies in FP32 only: far copies' node coordinates round differently, and the
curl form of the metrics multiplies two of them.)
"""
import numpy as np
import pytest

import oracle as O
import problems as PB
from test_gpu_fd_kernels import R, torch  # noqa: F401

pytestmark = pytest.mark.gpu


def points_of(torch, gm, warp):
    """Warped nodes of a unit-spaced brick, (K, dim, Np) on the device."""
    dim, nq = gm.cell.dim, gm.cell.nq
    c = torch.from_numpy(gm.cell_centres()).cuda()
    xi = torch.from_numpy(np.asarray(gm.cell.points_1d)).cuda()
    idx = torch.arange(nq ** dim, device="cuda")
    x = [c[:, d, None] + 0.5 * xi[(idx // nq ** d) % nq][None] for d in range(dim)]
    return torch.stack(warp(torch.sin, *x), 1).contiguous()


def warp_of(small):
    k = [2 * np.pi / n for n in small]

    def warp(sin, *x):  # periodic with the small brick
        d = len(x)
        return [x[j] + 0.04 * sin(k[(j + 1) % d] * x[(j + 1) % d]) for j in range(d)]
    return warp


# small brick, copies per direction; what the launch does beyond the caches
CASES = [
    # 3-D column kernel: a wave per cell (FP32 stages; Nq = 7), packed (others)
    (3, 5, "f64", "brick", "weak", "rusanov", [3, 2, 2], [9, 14, 13], False),
    (3, 5, "f32", "brick", "weak", "rusanov", [3, 2, 2], [11, 17, 17], False),
    (3, 5, "f32", "warp", "weak", "rusanov", [3, 2, 2], [11, 17, 17], False),
    (3, 6, "f64", "brick", "weak", "rusanov", [3, 2, 2], [8, 11, 11], True),
    (3, 6, "f32", "brick", "weak", "rusanov", [3, 2, 2], [9, 15, 15], False),
    (3, 6, "f32", "warp", "weak", "rusanov", [3, 2, 2], [9, 15, 15], False),
    (3, 7, "f64", "brick", "weak", "rusanov", [3, 2, 2], [6, 10, 10], False),
    (3, 7, "f32", "warp", "weak", "rusanov", [3, 2, 2], [8, 12, 12], False),
    # 2-D: streamed affine and curved cells
    (2, 6, "f64", "brick", "weak", "rusanov", [5, 3], [59, 99], True),
    (2, 6, "f32", "brick", "weak", "rusanov", [5, 3], [97, 139], False),
    (2, 4, "f64", "warp", "weak", "rusanov", [5, 3], [89, 149], True),
    # flux differencing: line kernel, node kernel
    (3, 8, "f64", "brick", "ec", "ec", [3, 2, 2], [6, 9, 8], True),
    (3, 5, "f32", "brick", "ec", "rusanov", [3, 2, 2], [11, 17, 17], True),
    (3, 4, "f32", "warp", "ec", "ec", [3, 2, 2], [15, 21, 21], True),
    (3, 6, "f64", "brick", "central", "rusanov", [3, 2, 2], [8, 11, 11], True),
]


@pytest.mark.parametrize("dim,nq,dtype,geometry,form,face,small,copies,streams", CASES)
def test_copies(torch, R, dim, nq, dtype, geometry, form, face, small, copies, streams):
    print(f"large grid dim={dim} nq={nq} {dtype} {geometry} {form} {small} x {copies}", flush=True)
    per, cell = (True,) * dim, R.LobattoCell(*([nq] * dim))
    warp = warp_of(small)
    coords = [np.arange(k + 1) * 1.0 for k in small]
    gms = [R.GridManager(cell, R.brick([np.arange(k + 1) * 1.0 for k in n], per))
           for n in (small, [a * b for a, b in zip(small, copies)])]
    # the small brick's cell that each large cell copies
    place = lambda c: tuple(np.floor(c).astype(int) % small)  # noqa: E731
    first = {place(c): e for e, c in enumerate(gms[0].cell_centres())}
    copy = torch.tensor([first[place(c)] for c in gms[1].cell_centres()], device="cuda")

    flux = {"rusanov": R.RusanovFlux, "ec": R.EntropyConservativeFlux}[face]()
    vol = {"weak": R.WeakForm(), "central": R.FluxDifferencingForm(R.CentralFlux()),
           "ec": R.FluxDifferencingForm(R.EntropyConservativeFlux())}[form]
    kw = dict(dtype=dtype, volume_form=vol)
    if geometry == "warp":
        dg = R.DGSEM.forest(gms[1], R.EulerLaw(dim), flux, points=points_of(torch, gms[1], warp), **kw)
    else:
        dg = R.DGSEM.brick(gms[1], R.EulerLaw(dim), flux, **kw)
    assert dg.info.state_bytes * 3 > 256 << 20 and dg.info.streaming == streams
    og = O.BrickGrid(nq, coords, per,
                     warp=(lambda *x: warp(np.sin, *x)) if geometry == "warp" else None)
    odg = O.DG(og, "euler", volume_flux=None if form == "weak" else form, surface_flux=face)

    rng = np.random.default_rng(nq)
    shape = (og.K, nq ** dim)
    rho, p = (1 + 0.2 * rng.uniform(-1, 1, shape) for _ in range(2))
    mom = [0.3 * rng.uniform(-1, 1, shape) for _ in range(dim)]
    q = np.stack([rho] + mom + [PB.euler_energy(rho, mom, p, 1.4)], axis=1)
    one = torch.from_numpy(q).to(dg.torch_dtype).cuda()
    qh = one.double().cpu().numpy().reshape(-1)
    L = np.zeros(q.size)
    odg.rhs(L, qh.copy(), 0.0, increment=False)
    d0 = torch.from_numpy(np.abs(L).max() * 0.1 * rng.uniform(-1, 1, q.shape)).to(dg.torch_dtype).cuda()
    qd = one[copy].contiguous()

    def check(got, want, bar, what):
        w = torch.from_numpy(want.reshape(q.shape)).cuda()
        err, size = 0.0, 0.0
        for a in range(0, dg.K, 4096):
            x = w[copy[a:a + 4096]]
            err += float(((got[a:a + 4096].double() - x) ** 2).sum())
            size += float((x ** 2).sum())
        print(f"   {what} {(err / size) ** 0.5:.2e}", flush=True)
        assert (err / size) ** 0.5 <= bar

    dq = dg.GridArray(0.0)
    dg(dq, qd, 0.0, increment=False)
    check(dq, L, 1e-12 if dtype == "f64" else 1e-4, "right-hand side")
    dq, qo = d0[copy].contiguous(), torch.empty_like(qd)
    dg.lsrk_stage(qo, qd, dq, -0.6, 1e-4)
    want = -0.6 * d0.double().cpu().numpy().reshape(-1) + L
    check(dq, want, 1e-12 if dtype == "f64" else 1e-4, "dq")
    check(qo, qh + 1e-4 * want, 1e-12 if dtype == "f64" else 1e-6, "q_out")


@pytest.mark.parametrize("dtype", ["f64", "f32"])
@pytest.mark.parametrize("nq", [5, 6, 7])
def test_one_cell(torch, R, nq, dtype):
    print(f"one 3-D cell nq={nq} {dtype}", flush=True)
    coords, per = [np.array([0.0, 1.0])] * 3, (False,) * 3
    grid = R.generate(R.GridManager(R.LobattoCell(nq, nq, nq), R.brick(coords, per)))
    dg = R.DGSEM(law=R.EulerLaw(3), grid=grid, dtype=dtype)
    og = O.BrickGrid(nq, coords, per)
    q = PB.euler_wave(og.point_fields(), 3, 0.0)
    qd = torch.from_numpy(q).to(dg.torch_dtype).cuda().reshape(dg.K, dg.ns, dg.Np).contiguous()
    want = np.zeros(q.size)
    O.DG(og, "euler").rhs(want, qd.double().cpu().numpy().reshape(-1).copy(), 0.0, increment=False)
    dq = dg.GridArray(0.0)
    dg(dq, qd, 0.0, increment=False)
    dg.synchronize()
    got = dq.double().cpu().numpy().reshape(-1)
    assert np.linalg.norm(got - want) <= (1e-12 if dtype == "f64" else 1e-4) * np.linalg.norm(want)
