"""Oriented and explicit faces through every stage kernel (needs an MI355X).

A brick's faces all have the same orientation.  Here the neighbours of a
library-made brick are redrawn at random, the same for the oracle: a face takes
another cell's face with its nodes reversed, swapped or both (a record with an
orientation), or a random set of nodes (explicit indices).  What the operator
then means does not matter: q+ = q[vmapP] on both sides.  FP64 1e-12, FP32 1e-4.
"""
import numpy as np
import pytest

import oracle as O
import problems as PB
from test_gpu_fd_kernels import R, extents, rel_l2, states, torch  # noqa: F401

pytestmark = pytest.mark.gpu


def redraw(vmapP, dim, nq, rng):
    """Half of the faces oriented, a third of the rest explicit."""
    K, nfpt = vmapP.shape
    nfp = nfpt // (2 * dim)
    node = np.arange(nq ** dim).reshape((nq,) * dim)  # axes from the last direction
    out = vmapP.copy()
    for e in range(K):
        for f in range(2 * dim):
            pick = rng.uniform()
            if pick < 0.5:
                g, cell = rng.integers(2 * dim), rng.integers(K)
                face = np.take(node, 0 if g % 2 == 0 else nq - 1, axis=dim - 1 - g // 2)
                if dim == 3 and rng.uniform() < 0.5:
                    face = face.T
                for axis in range(dim - 1):
                    if rng.uniform() < 0.5:
                        face = np.flip(face, axis)
                new = face.reshape(-1) + nq ** dim * cell + 1
            elif pick < 0.67:
                new = rng.integers(1, K * nq ** dim + 1, nfp)
            else:
                continue
            out[e, f * nfp:(f + 1) * nfp] = new
    return out


def warp2(x, y):
    return x + 0.02 * np.sin(np.pi * y), y + 0.02 * np.sin(np.pi * x)


def warp3(x, y, z):
    return x + 0.02 * np.sin(np.pi * y), y + 0.02 * np.sin(np.pi * z), z + 0.02 * np.sin(np.pi * x)


FORMS = [("weak", "rusanov"), ("central", "rusanov"), ("ec", "ec"), ("ec", "rusanov")]
CASES = [(dim, nq, geometry, form, face, False)
         for dim, nq in ((1, 4), (2, 5), (3, 4), (3, 6)) for geometry in ("auto", "warp")
         for form, face in FORMS if dim > 1 or geometry == "auto"]
CASES += [(2, 5, "auto", "ec", "rusanov", True), (2, 8, "warp", "ec", "ec", True),
          (3, 4, "warp", "ec", "rusanov", True), (3, 6, "auto", "ec", "ec", True)]


@pytest.mark.parametrize("dtype", ["f64", "f32"])
@pytest.mark.parametrize("dim,nq,geometry,form,face,line", CASES)
def test_rhs(torch, R, dim, nq, geometry, form, face, line, dtype):
    n = extents(dim, nq, dtype, True) if line else [7, 3, 2][:dim]
    print(f"face maps dim={dim} nq={nq} {geometry} {form} {face} {dtype} cells={n}", flush=True)
    coords, per = [PB.julia_range(0, 1, k + 1) for k in n], (False,) * dim
    warp = {2: warp2, 3: warp3}[dim] if geometry == "warp" else None
    grid = R.generate(R.GridManager(R.LobattoCell(*([nq] * dim)), R.brick(coords, per)), warp=warp)
    og = O.BrickGrid(nq, coords, per, warp=warp)
    rng = np.random.default_rng(dim * 10 + nq)
    grid.vmapP = redraw(np.asarray(grid.vmapP).reshape(og.K, -1), dim, nq, rng)
    grid.boundarycodes = np.zeros_like(np.asarray(grid.boundarycodes))
    og.vmapP, og.bc = np.ascontiguousarray(grid.vmapP).reshape(-1), np.zeros_like(og.bc)
    flux = {"rusanov": R.RusanovFlux, "ec": R.EntropyConservativeFlux}[face]()
    vol = {"weak": R.WeakForm(), "central": R.FluxDifferencingForm(R.CentralFlux()),
           "ec": R.FluxDifferencingForm(R.EntropyConservativeFlux())}[form]
    dg = R.DGSEM(law=R.EulerLaw(dim), grid=grid, dtype=dtype, surface_numericalflux=flux,
                 volume_form=vol)
    assert dg.info.faces_explicit > 0
    odg = O.DG(og, "euler", volume_flux=None if form == "weak" else form, surface_flux=face)
    q = states(og.point_fields(), dim, 5)
    qd = torch.from_numpy(q).to(dg.torch_dtype).cuda().reshape(dg.K, dg.ns, dg.Np).contiguous()
    want = np.zeros(q.size)
    odg.rhs(want, qd.double().cpu().numpy().reshape(-1).copy(), 0.0, increment=False)
    dq = dg.GridArray(0.0)
    dg(dq, qd, 0.0, increment=False)
    dg.synchronize()
    err = rel_l2(dq.double().cpu().numpy().reshape(-1), want)
    print(f"   dq {err:.2e}", flush=True)
    assert err <= (1e-12 if dtype == "f64" else 1e-4)


@pytest.mark.parametrize("dim,nq,form", [(2, 4, "weak"), (2, 4, "ec"), (3, 3, "ec"), (3, 3, "weak")])
def test_fp32_geometry_copies(torch, R, dim, nq, form):
    """An FP32 handle of curved cells holds, beyond the FP64 handle's arrays, the
    copies its stages read: metric terms, 1 / MJ and faces, and MJ where the
    weak form's 3-D relaxation stage reads it."""
    n = [3, 2, 2][:dim]
    grid = R.generate(R.GridManager(R.LobattoCell(*([nq] * dim)), R.brick(
        [PB.julia_range(0, 1, k + 1) for k in n], (False,) * dim)), warp={2: warp2, 3: warp3}[dim])
    vol = R.WeakForm() if form == "weak" else R.FluxDifferencingForm(R.EntropyConservativeFlux())
    held = []
    for dtype in ("f32", "f64"):
        dg = R.DGSEM(law=R.EulerLaw(dim), grid=grid, dtype=dtype, volume_form=vol,
                     surface_numericalflux=R.RusanovFlux())
        held.append(dg.info.device_bytes)
    copies = dg.K * (dg.Np * (dim * dim + 1) + 2 * dim * (dim + 1) * nq ** (dim - 1))
    if form == "weak" and dim == 3:
        copies += dg.K * dg.Np
    tables = 0 if form == "weak" else 2 * nq * nq  # pair weights, in the state's type
    assert held[0] - held[1] == 4 * (copies - tables)
