"""The fixed-length complex64 BiCGStab inside the mixed-precision solve
(inner_tol = 0), against the iteration written out pass by pass.

solve_mixed with one outer step returns x = c z for the inner solution z and
one complex number c.  The reference keeps every vector in complex64, forms
every update and every scalar in complex128 and rounds each vector once; its
matvecs are single complex64 applications (Helm3d.apply).  The right-hand side
has entries +-1 +-i at 2^13 points, so its norm is a power of two and the inner
solve starts from exactly b / |b|.

Bar: z is stored in complex64, one rounding of at most 2^-24 of each part, so
|x - c z| <= 2^-24 |c z| (roundings average to about 0.4 of the bound).  Vector
updates in single precision, or with scalars rounded to single precision, miss
it.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _dot(a, b):
    import torch
    return torch.vdot(a.to(torch.complex128), b.to(torch.complex128))


def _reference(H, b, its, adjoint):
    """z of `its` BiCGStab iterations from z = 0 with rhat = b (complex64);
    the last update is returned unrounded."""
    import torch
    up, down = (lambda a: a.to(torch.complex128)), (lambda a: a.to(torch.complex64))
    r, p, z, rho = b, b, torch.zeros_like(b), _dot(b, b)
    for it in range(its):
        v = H.apply(p, adjoint=adjoint)
        alpha = rho / _dot(b, v)
        s64 = up(r) - alpha * up(v)
        s = down(s64)
        t = H.apply(s, adjoint=adjoint)
        omega = _dot(t, s) / _dot(t, t)
        if it == its - 1:
            return up(z) + alpha * up(p) + omega * s64
        z = down(up(z) + alpha * up(p) + omega * up(s))
        r64 = up(s) - omega * up(t)
        r = down(r64)
        new = _dot(b, r64)
        beta = (new / rho) * (alpha / omega)
        p = down(up(r) + beta * (up(p) - omega * up(v)))
        rho = new


@pytest.mark.parametrize("n", [(33, 27, 22), (97, 41, 30)])
@pytest.mark.parametrize("wnc", [False, True])
@pytest.mark.parametrize("mode", [1, 2])
@pytest.mark.parametrize("its", [2, 3])
def test_fixed_inner_solve_rounds_each_vector_once(n, wnc, mode, its):
    import torch
    from helm3d import Helm3d
    print(f"fixed inner solve n={n} wnc={wnc} mode={mode} its={its}", flush=True)
    rng = np.random.default_rng(41)
    N = int(np.prod(n))
    wn = (2 * np.pi * 6.0 / rng.uniform(1800.0, 4300.0, N)) ** 2
    if wnc:
        wn = wn * (1.0 + 0.02j)
    dev = torch.device("cuda:0")
    H = Helm3d(n, (20.0,) * 3, np.full((2, 3), 5), torch.from_numpy(wn).to(dev))
    b = np.zeros(N, complex)
    at = rng.choice(N, 2 ** 13, replace=False)
    b[at] = rng.choice([-1.0, 1.0], at.size) + 1j * rng.choice([-1.0, 1.0], at.size)
    b = torch.from_numpy(b).to(dev)
    x, _ = H.solve_mixed(b, mode=mode, tol=1e-30, maxinnerit=1, maxit=2, inner_tol=0.0, inner_maxit=its)
    z = _reference(H, (b / 128.0).to(torch.complex64), its, mode != 1)
    cz = (_dot(z, x) / _dot(z, z)) * z
    err = float((x - cz).norm() / cz.norm())
    print(f"  err {err:.3e} (bar {2.0 ** -24:.3e})", flush=True)
    assert float(cz.norm()) > 0.0 and err <= 2.0 ** -24
