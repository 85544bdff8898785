"""Interior displacements do not depend on which other points are in the set, how many there are or in
which order they come: sets of 1 .. 130 points (edges of the 16-point waves), reversed, with a point
twice, and points on a node (which take the node's displacement) against one set of all of them.

Bar: 1e-12 of the largest component: only the order of at most ~2e4 additions of similar size differs
(1e4 eps at the worst, their square root in practice)."""
import numpy as np
import pytest

from multifebe_amd import mesh as M

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("harmonic", [False, True])
def test_points_sets(harmonic):
    from multifebe_amd import bem
    bem._torch()
    m = M.pressure_hemisphere_bcs(M.sphere(6))
    s = bem.BemSystem(m)
    rng = np.random.default_rng(3)
    u = rng.standard_normal((m.nn, 3)) * 1e-3
    t = rng.standard_normal((m.nn, 3)) * 1e6
    mu, mu_c, lam_c = M.elastic_constants(1e9, 0.3, 0.05)
    if harmonic:
        u, t = u * (1 + 0.5j), t * (1 - 0.3j)
        kw = dict(omega=2.0 * np.sqrt(mu / 2000.0), lam=lam_c, mu_c=mu_c, rho=2000.0)
    else:
        kw = dict(mu=mu, nu=0.3)
    x = M.points_off_surface(m, 128, 0.02, 0.8, seed=4, outward=False)
    x = np.concatenate([x, m.x[[5]], x[[7]]])

    def field(pts):
        return s.points(np.ascontiguousarray(pts)).displacement(u, t, **kw).cpu().numpy()
    ref = field(x)
    tol = 1e-12 * np.abs(ref).max()
    assert np.array_equal(ref[128], u[5]) and np.abs(ref[129] - ref[7]).max() <= tol
    for n in (1, 15, 16, 17, 63, 64, 65, 130):
        assert np.abs(field(x[:n]) - ref[:n]).max() <= tol, n
    assert np.abs(field(x[::-1]) - ref[::-1]).max() <= tol


def test_boundary_fields_on_the_gpu():
    """Device tensors give what numpy arrays of the same values give, in any plain type and stride;
    lazily conjugated ones give their values, tensors that require gradients are refused."""
    import torch
    from multifebe_amd import bem
    m = M.pressure_hemisphere_bcs(M.sphere(4))
    mu, mu_c, lam_c = M.elastic_constants(1e9, 0.3, 0.05)
    kw = dict(omega=2.0 * np.sqrt(mu / 2000.0), lam=lam_c, mu_c=mu_c, rho=2000.0)
    p = bem.BemSystem(m).points(M.points_off_surface(m, 20, 0.02, 0.8, seed=4, outward=False))
    rng = np.random.default_rng(5)
    u, t = (rng.standard_normal((m.nn, 3)) * (1 + 0.5j) for _ in range(2))
    ref = p.displacement(u, t, **kw)
    ud, td = torch.from_numpy(u).cuda(), torch.from_numpy(t).cuda()
    assert torch.allclose(p.displacement(ud, td, **kw), ref, rtol=0, atol=1e-13 * ref.abs().max())
    ut = ud.T.contiguous().T
    assert torch.allclose(p.displacement(ut, td, **kw), ref, rtol=0, atol=1e-13 * ref.abs().max())
    lazy = p.displacement(torch.from_numpy(u.conj()).cuda().conj(), td, **kw)
    assert torch.allclose(lazy, ref, rtol=0, atol=1e-13 * ref.abs().max())
    with pytest.raises(RuntimeError):
        p.displacement(ud.clone().requires_grad_(), td, **kw)
