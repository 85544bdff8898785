"""Assembly under every kind of boundary condition an element can have: traction-free (t* alone is
integrated), held at zero (u* alone), and everything that needs both, on closed and open surfaces,
against the oracle.  Bar: 1e-10 of the largest entry of the row (A) and of max |b| (b), the bar of the
whole-boundary assemblies; b is exactly zero without prescribed values."""
import numpy as np
import pytest

from multifebe_amd import mesh as M

pytestmark = pytest.mark.gpu


def _conditions(m, kind, rng):
    ct, cv = np.zeros((m.nn, 3), np.int32), np.zeros((m.nn, 3))
    if kind == "free":
        ct[:] = 1
    elif kind == "moved":
        cv[:] = rng.uniform(-1, 1, cv.shape)
    elif kind == "loaded":
        ct[:] = 1
        cv[:] = rng.uniform(-1e6, 1e6, cv.shape)
    elif kind == "halves":          # elements of each single kind and mixed ones between them
        ct[m.x[:, 0] > np.median(m.x[:, 0])] = 1
    elif kind == "mixed":
        ct[:] = rng.choice([0, 1, 10], ct.shape)
        cv[:] = np.where(rng.random(cv.shape) < 0.5, 0.0, np.where(ct == 0, 1e-3, 1e6))
    m.ctype, m.cval = ct, cv
    return m


@pytest.mark.parametrize("surface", ["cube", "sphere", "open"])
@pytest.mark.parametrize("kind", ["fixed", "free", "moved", "loaded", "halves", "mixed"])
def test_conditions(oracle, surface, kind):
    from multifebe_amd import bem
    bem._torch()
    m = {"cube": lambda: M.cube(4), "sphere": lambda: M.sphere(4),
         "open": lambda: M.free_surface(4.0, 4, 2.0)}[surface]()
    m = _conditions(m, kind, np.random.default_rng(5))
    mu, mu_c, lam_c = M.elastic_constants(1e9, 0.3, 0.05)
    s = bem.BemSystem(m)
    for omega in (None, 1.3 * np.sqrt(mu / 2000.0)):
        if omega is None:
            At, b = s.assemble_staela(mu, 0.3)
            Ao, bo = oracle.assemble(m, mu=mu, nu=0.3)
        else:
            At, b = s.assemble_harela(omega, lam_c, mu_c, 2000.0, 0.3)
            Ao, bo = oracle.assemble(m, lam_c=lam_c, mu_c=mu_c, rho=2000.0, omega=omega, nu=0.3)
        A, b = At.T.cpu().numpy(), b.cpu().numpy()
        assert np.max(np.abs(A - Ao) / np.abs(Ao).max(axis=1, keepdims=True)) <= 1e-10
        if np.any(m.cval):
            assert np.abs(b - bo).max() <= 1e-10 * np.abs(bo).max()
        else:
            assert not b.any()
