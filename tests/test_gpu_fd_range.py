"""The entropy-conservative stage far from values of order one (needs an MI355X).

Euler's equations scale: with density, momentum and energy times S = 2^k every
term of the right-hand side is times S, and with velocities times s = 2^m and
pressure times s^2 the rows of the right-hand side are times s (density), s^2
(momentum) and s^3 (energy).  So the operator on a scaled state is the scaled
operator on values of order one, against the oracle there at the bars of
test_gpu_fluxdiff.py (FP64 1e-12, FP32 1e-4).  Neighbouring nodes differ by
a factor of about five (the means need logarithms), and the scales put the
squares of densities, or of rho / p, past either end of the type's range.
Momentum squared stays inside it.
"""
import numpy as np
import pytest

import oracle as O
import problems as PB
from test_gpu_fd_kernels import R, extents, make, rel_l2, torch  # noqa: F401

pytestmark = pytest.mark.gpu


def states(P, dim, nq, what, seed):
    """Every line alternates between values near 0.9 and near 0.2 of the scaled
    quantity (density, or b = rho / p); the other one hardly varies."""
    rng = np.random.default_rng(seed)
    shape = P[:, 0, :].shape
    node = np.arange(nq ** dim)
    odd = sum(node // nq ** d % nq for d in range(dim)) % 2
    far = np.where(odd, rng.uniform(0.85, 1.0, shape), rng.uniform(0.17, 0.22, shape))
    near = 1 + 1e-3 * rng.uniform(-1, 1, shape)
    rho, b = (far, near) if what == "rho" else (near, far)
    return rho, [0.1 * rng.uniform(-1, 1, shape) for _ in range(dim)], rho / b


@pytest.mark.parametrize("line", [True, False])
@pytest.mark.parametrize("what", ["rho", "velocity"])
@pytest.mark.parametrize("sign", [1, -1])
@pytest.mark.parametrize("dim,nq,geometry,face,dtype", [
    (2, 5, "auto", "ec", "f64"), (2, 4, "general", "rusanov", "f32"),
    (3, 4, "auto", "rusanov", "f32"), (3, 6, "general", "ec", "f64"), (3, 3, "auto", "ec", "f32")])
def test_scaled_state(torch, R, dim, nq, geometry, face, dtype, sign, what, line):
    n = extents(dim, nq, dtype, line)
    print(f"fd range dim={dim} nq={nq} {geometry} {face} {dtype} {what} {sign} cells={n}", flush=True)
    dg, og, odg = make(R, dim, nq, n, dtype, geometry, face, (True,) * dim)
    rho, u, p = states(og.point_fields(), dim, nq, what, 5)
    half = 32 if dtype == "f32" else 256  # the type's range is 2^(4 half)
    S, s = (2.0 ** (2 * half * sign), 1.0) if what == "rho" else (1.0, 2.0 ** (half * sign))

    def pack(S, s):
        mom = [rho * v for v in u]
        E = PB.euler_energy(rho, mom, p, 1.4)
        return np.stack([S * rho] + [S * s * m for m in mom] + [S * s * s * E], axis=1)
    # rounded to the type at order one, then scaled (both exact)
    q1 = torch.from_numpy(pack(1.0, 1.0)).to(dg.torch_dtype).double().numpy()
    rows = np.array([1.0] + [s] * dim + [s * s])[None, :, None] * S
    qd = torch.from_numpy(q1 * rows).to(dg.torch_dtype).cuda().contiguous()
    want = np.zeros(q1.size)
    odg.rhs(want, np.ascontiguousarray(q1).reshape(-1), 0.0, increment=False)
    dq = dg.GridArray(0.0)
    dg(dq, qd, 0.0, increment=False)
    dg.synchronize()
    got = dq.double().cpu().numpy() / rows / s
    err = rel_l2(got.reshape(-1), want)
    print(f"   dq {err:.2e}", flush=True)
    assert err <= (1e-12 if dtype == "f64" else 1e-4)


@pytest.mark.parametrize("line", [True, False])
@pytest.mark.parametrize("dim,nq,geometry,face,dtype", [
    (1, 4, "auto", "ec", "f64"), (2, 5, "auto", "rusanov", "f64"), (3, 4, "general", "ec", "f32")])
def test_zero_pressure(torch, R, dim, nq, geometry, face, dtype, line):
    """A node of zero pressure (rho / p infinite): the flux's pressure average is
    zero and its logarithmic mean is not a number, so the energy of the node's
    lines is lost and density and momentum are not, as in the oracle."""
    if dim == 1 and line:
        pytest.skip("1-D has no line kernel")
    n = extents(dim, nq, dtype, line)
    print(f"fd zero pressure dim={dim} nq={nq} {geometry} {face} {dtype} cells={n}", flush=True)
    dg, og, odg = make(R, dim, nq, n, dtype, geometry, face, (True,) * dim)
    rho, u, p = states(og.point_fields(), dim, nq, "rho", 5)
    q = np.stack([rho] + [rho * v for v in u] + [PB.euler_energy(rho, [rho * v for v in u], p, 1.4)],
                 axis=1)
    at = (dg.K // 2, slice(None), nq ** dim // 2)
    q[at] = [1.0] + [0.0] * (dim + 1)
    qd = torch.from_numpy(q).to(dg.torch_dtype).cuda().contiguous()
    qh = qd.double().cpu().numpy()
    want = np.zeros(q.size)
    odg.rhs(want, np.ascontiguousarray(qh).reshape(-1), 0.0, increment=False)
    dq = dg.GridArray(0.0)
    dg(dq, qd, 0.0, increment=False)
    dg.synchronize()
    got = dq.double().cpu().numpy().reshape(-1)
    lost = ~np.isfinite(want)
    assert lost.any() and np.array_equal(lost, ~np.isfinite(got))
    err = rel_l2(got[~lost], want[~lost])
    print(f"   dq {err:.2e}", flush=True)
    assert err <= (1e-12 if dtype == "f64" else 1e-4)
