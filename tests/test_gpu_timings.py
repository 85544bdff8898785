"""timings(): near pairs and free terms share one launch, whose time is adaptive_ms; time_groups() has
each group launched and timed by itself, with the same matrix and statistics."""
import pytest

from multifebe_amd import mesh as M

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", ["cylinder", "open"])
@pytest.mark.parametrize("harmonic", [False, True])
def test_groups(shape, harmonic):
    from multifebe_amd import bem
    bem._torch()
    m = M.cylinder(4) if shape == "cylinder" else M.free_surface(4.0, 4, 2.0)
    M.pressure_hemisphere_bcs(m)
    mu, mu_c, lam_c = M.elastic_constants(1e9, 0.3, 0.05)
    s = bem.BemSystem(m)

    def assemble():
        At, b = (s.assemble_harela(900.0, lam_c, mu_c, 2000.0, 0.3) if harmonic
                 else s.assemble_staela(mu, 0.3))
        return At, b, s.timings(), s.stats()
    A0, b0, t0, st0 = assemble()
    assert t0["singular_ms"] == 0.0 and t0["adaptive_ms"] > 0 and t0["regular_ms"] > 0
    s.time_groups()
    A1, b1, t1, st1 = assemble()
    assert min(t1[k] for k in ("regular_ms", "adaptive_ms", "singular_ms", "freeterm_zero_ms")) > 0
    s.time_groups(False)
    A2, b2, t2, st2 = assemble()
    assert t2["singular_ms"] == 0.0 and st0 == st1 == st2
    for A, b in ((A1, b1), (A2, b2)):
        # only the order of a few additions differs
        assert (A - A0).abs().max() <= 1e-14 * A0.abs().max()
        assert (b - b0).abs().max() <= 1e-14 * b0.abs().max()
