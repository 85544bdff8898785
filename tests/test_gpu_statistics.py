"""Quadrature points and leaves that stats() reports: nothing of the adaptive and singular pairs before
an assembly has run (capturing a batch runs none), those of one assembly after one, and after a batch
those of every job of the mesh, subdivided pairs and single leaves alike."""
import pytest

from multifebe_amd import mesh as M

pytestmark = pytest.mark.gpu


def near(s):
    st = s.stats()
    return st["points"] - st["regular_points"], st["leaves"]


@pytest.mark.parametrize("shape", ["slab", "cylinder", "open"])
def test_points_and_leaves(shape):
    import torch
    from multifebe_amd import bem
    bem._torch()
    m = {"slab": lambda: M.slab(0.25, 1.0, 0.02), "cylinder": lambda: M.cylinder(4),
         "open": lambda: M.free_surface(4.0, 4, 2.0)}[shape]()
    M.pressure_hemisphere_bcs(m)
    mu, mu_c, lam_c = M.elastic_constants(1e9, 0.3, 0.05)
    p = dict(lam=lam_c, rho=2000.0, nu=0.3)
    omega = 1.3 * (mu / 2000.0) ** 0.5
    one = bem.BemSystem(m)
    assert near(one) == (0, 0)
    for _ in range(2):
        one.assemble_harela(omega, lam_c, mu_c, 2000.0, 0.3)
        points, leaves = near(one)
        assert points >= 25 * leaves and leaves >= one.stats()["adaptive"] > 0
    if shape == "slab":   # subdivided pairs among them
        assert leaves > one.stats()["adaptive"]
    assert one.stats()["singular"] > 0 and points > 25 * leaves
    first = points, leaves

    s = bem.BemSystem(m)
    jobs = []
    for k in range(3):
        At, b = s.alloc(True)
        jobs.append(dict(system=s, At=At, b=b, omega=omega * (1 + k), mu_c=mu_c, **p))
    g = bem.BatchGraph(jobs)
    torch.cuda.synchronize()
    assert near(s) == (0, 0)
    for _ in range(2):
        g.launch()
        g.check()
        assert near(s) == (3 * first[0], 3 * first[1])
    bem.assemble_batch(jobs[:2])
    assert near(s) == (2 * first[0], 2 * first[1])
    s.assemble_staela(mu, 0.3)
    assert near(s) == first
