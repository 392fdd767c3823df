"""The two decompositions of the flux-differencing stage (needs an MI355X).

Large grids with the entropy-conservative flux run a lane per line of a cell,
the others a lane per node; the line kernel picks a short or a long series, or
the logarithm, for its logarithmic means by the line's extremes.  Grids just
above the switch (with remainders in every workgroup size) and far below it,
states whose lines need each of the three, against the oracle at the bars of
test_gpu_fluxdiff.py (FP64 1e-12, FP32 right-hand sides 1e-4).
"""
import ctypes
import math

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


# cells per workgroup and waves of the line kernel
CELLS = {2: 16, 3: 7, 4: 4, 5: 3, 6: 1, 7: 1, 8: 1}


def extents(dim, nq, dtype, line):
    """A brick just above the switch to the line kernel, or a small one."""
    if not line:
        return [5, 3, 4][:dim]
    c = 32 // nq if dim == 2 else CELLS[nq]
    waves = -(-(c * dim * nq ** (dim - 1)) // 64)
    need = (1152 if dtype == "f64" else 1792) * c // waves + 1
    n = [int(need ** (1 / dim)) + 1] * dim
    n[0] += 2
    # no multiple of the workgroup's cells
    return [next(k for k in range(v, v + 16) if math.gcd(k, c) == 1) for v in n]


def states(P, dim, seed):
    """Density and pressure noise of amplitude 1e-4, 0.05 and 0.5 in thirds of
    the domain along x: short series, long series, logarithms."""
    rng = np.random.default_rng(seed)
    x = P[:, 0, :]
    amp = np.where(x < 1 / 3, 1e-4, np.where(x < 2 / 3, 0.05, 0.5))
    rho = 1 + amp * rng.uniform(-1, 1, x.shape)
    p = 1 + amp * rng.uniform(-1, 1, x.shape)
    mom = [rho * rng.uniform(-0.3, 0.3, x.shape) for _ in range(dim)]
    E = PB.euler_energy(rho, mom, p, 1.4)
    return np.ascontiguousarray(np.stack([rho] + mom + [E], axis=1)).reshape(-1)


def make(R, dim, nq, n, dtype, geometry, face, per, directions=None):
    coords = [PB.julia_range(0, 1, k + 1) for k in n]
    grid = R.generate(R.GridManager(R.LobattoCell(*([nq] * dim)), R.brick(coords, per)))
    ec = R.EntropyConservativeFlux()
    dg = R.DGSEM(law=R.EulerLaw(dim), grid=grid, dtype=dtype, geometry=geometry,
                 surface_numericalflux=ec if face == "ec" else R.RusanovFlux(),
                 volume_form=R.FluxDifferencingForm(ec), directions=directions)
    og = O.BrickGrid(nq, coords, per)
    return dg, og, O.DG(og, "euler", volume_flux="ec", surface_flux=face)


@pytest.mark.parametrize("line", [True, False])
@pytest.mark.parametrize("dtype", ["f64", "f32"])
@pytest.mark.parametrize("dim,nq,geometry,face", [
    (2, 2, "auto", "ec"), (2, 3, "general", "rusanov"), (2, 5, "auto", "rusanov"),
    (2, 6, "general", "ec"), (2, 7, "auto", "ec"), (2, 8, "general", "rusanov"),
    (3, 2, "general", "ec"), (3, 3, "auto", "rusanov"), (3, 4, "auto", "ec"),
    (3, 5, "general", "rusanov"), (3, 6, "auto", "rusanov"), (3, 7, "general", "ec"),
    (3, 7, "auto", "rusanov"), (3, 8, "auto", "ec"), (3, 8, "general", "rusanov")])
def test_stage_matches_oracle(torch, R, dim, nq, geometry, face, dtype, line):
    n = extents(dim, nq, dtype, line)
    print(f"fd kernels dim={dim} nq={nq} {geometry} {face} {dtype} cells={n}", flush=True)
    per = (True, False, True)[:dim]
    dg, og, odg = make(R, dim, nq, n, dtype, geometry, face, per)
    q = states(og.point_fields(), dim, 5)
    qd = torch.from_numpy(q).to(dg.torch_dtype).cuda().reshape(dg.K, dg.ns, dg.Np).contiguous()
    qh = qd.double().cpu().numpy().reshape(-1).copy()
    L = np.zeros(q.size)
    odg.rhs(L, qh, 0.0, increment=False)
    dq0 = 0.1 * np.abs(L).max() * np.random.default_rng(6).uniform(-1, 1, q.size)
    dqd = torch.from_numpy(dq0).to(dg.torch_dtype).cuda().reshape(qd.shape).contiguous()
    dqh = dqd.double().cpu().numpy().reshape(-1)
    qo = torch.empty_like(qd)
    a, bdt = -0.6, 1e-4
    dg.lsrk_stage(qo, qd, dqd, a, bdt)
    dg.synchronize()
    want = a * dqh + L
    e1 = rel_l2(dqd.double().cpu().numpy().reshape(-1), want)
    e2 = rel_l2(qo.double().cpu().numpy().reshape(-1), qh + bdt * want)
    print(f"   dq {e1:.2e}, q_out {e2:.2e}", flush=True)
    assert e1 <= (1e-12 if dtype == "f64" else 1e-4)
    assert e2 <= (1e-12 if dtype == "f64" else 1e-6)


@pytest.mark.parametrize("dim,nq", [(2, 6), (3, 8)])
def test_line_kernel_directions_add_up(torch, R, dim, nq):
    """L(all) = L(one direction) + L(the others)."""
    n = extents(dim, nq, "f64", True)
    print(f"fd line kernel directions dim={dim} nq={nq} cells={n}", flush=True)
    per = (True,) * dim
    out = []
    for dirs in (None, [1], list(range(2, dim + 1))):
        dg, og, _ = make(R, dim, nq, n, "f64", "auto", "rusanov", per, directions=dirs)
        q = states(og.point_fields(), dim, 7)
        qd = torch.from_numpy(q).cuda().reshape(dg.K, dg.ns, dg.Np).contiguous()
        dq = dg.GridArray(0.0)
        dg(dq, qd, 0.0, increment=False)
        dg.synchronize()
        out.append(dq.cpu().numpy().reshape(-1))
    assert rel_l2(out[1] + out[2], out[0]) <= 1e-12


@pytest.mark.parametrize("dim,nq", [(2, 5), (3, 7)])
def test_line_kernel_relaxation_step(torch, R, dim, nq):
    """One RLSRK54 step through the line kernel's relaxation stages."""
    n = extents(dim, nq, "f64", True)
    print(f"fd line kernel relaxation dim={dim} nq={nq} cells={n}", flush=True)
    per = (True,) * dim
    dg, og, odg = make(R, dim, nq, n, "f64", "auto", "ec", per)
    q = states(og.point_fields(), dim, 9)
    dt = 0.05 / max(n) / nq ** 2
    qd = torch.from_numpy(q).cuda().reshape(dg.K, dg.ns, dg.Np).contiguous()
    solver = R.RLSRK54(dg, qd, dt)
    R.dostep_(qd, solver)
    want, g = q.copy(), ctypes.c_double(1.0)
    z = [np.zeros(q.size) for _ in range(3)]
    O.lib().orc_dg_rlsrk_step(odg.h, 54, want, *z, 0.0, dt, ctypes.byref(g))
    got = qd.cpu().numpy().reshape(-1)
    print(f"   q {rel_l2(got, want):.2e}, gamma {solver.gamma!r} vs {g.value!r}", flush=True)
    # the step's change, and the relaxation parameter to the residual's bound
    # of 10 eps over its slope: gamma enters the step's change linearly
    assert rel_l2(got - q, want - q) <= 1e-9
    assert rel_l2(got, want) <= 1e-12
