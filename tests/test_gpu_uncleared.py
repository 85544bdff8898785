"""Assembly into buffers that hold NaN: the matrix is not cleared beforehand, so every entry has to be
stored by some element.  Closed and open surfaces, boundaries with a node that no element uses, with an
element that holds a node three times (a quadrilateral collapsed to a triangle on the open edge) -- which
are cleared and added to instead -- padded columns, the learned rules and captured batches.

Bars: 1e-10 of the largest entry of the row against the oracle, the bar of the whole-boundary
assemblies.  A node that no element uses is collocated as a point off the surface; the oracle leaves its
rows out, so they are held against its interior points.  The collapsed boundary is held against the same
geometry with three nodes in one place: its matrix is that one's with their rows and columns added, but
for the order of the additions (1e-12); the collapsed element's own rows are left out, its polar points
at the collapsed corner have no normal."""
import ctypes as C
import os

import numpy as np
import pytest

from multifebe_amd import mesh as M

pytestmark = pytest.mark.gpu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
NAN = float("nan")


def _mesh(kind):
    m = M.free_surface(4.0, 4, 2.0) if "open" in kind else M.sphere(4)
    x = np.concatenate([m.x, [[3.0, 2.5, 2.0]]]) if "unused" in kind else m.x
    return _conditions(x, m.conn)


def _conditions(x, conn):
    m = M.Mesh(x=np.ascontiguousarray(x), conn=np.ascontiguousarray(conn))
    rng = np.random.default_rng(2)
    m.ctype = np.ones((m.nn, 3), np.int32)
    m.ctype[m.x[:, 1] > 0.5] = 0
    m.cval = rng.uniform(-1, 1, (m.nn, 3)) * np.where(m.ctype == 0, 1e-3, 1e6)
    return m


def _collapsed():
    """(collapsed boundary, the same with nodes of their own in one place, where each of these goes)"""
    m = M.free_surface(4.0, 4, 2.0)
    e = m.conn[0]
    assert np.all(m.x[e[[0, 3, 7]], 0] == -2.0)      # an edge on the perimeter
    x = m.x.copy()
    x[e[[3, 7]]] = x[e[0]]
    split = _conditions(x, m.conn)
    split.ctype[e[[3, 7]]], split.cval[e[[3, 7]]] = split.ctype[e[0]], split.cval[e[0]]
    keep = np.setdiff1d(np.arange(m.nn), e[[3, 7]])
    to = np.full(m.nn, -1)
    to[keep] = np.arange(keep.size)
    to[e[[3, 7]]] = to[e[0]]
    c = M.Mesh(x=np.ascontiguousarray(x[keep]), conn=to[m.conn].astype(np.int32))
    c.ctype, c.cval = split.ctype[keep].copy(), split.cval[keep].copy()
    return c, split, to


KINDS = ["closed", "open", "unused closed", "unused open"]
MU, MU_C, LAM_C = M.elastic_constants(1e9, 0.3, 0.05)
OMEGA = 1.3 * np.sqrt(MU / 2000.0)


def _assemble(s, harmonic, pad=0):
    """twice into buffers that hold NaN: A, b and what lies between the columns"""
    import torch
    from multifebe_amd._lib import check, lib
    n, dt = s.n_dof, torch.complex128 if harmonic else torch.float64
    At = torch.empty((n, n + pad), dtype=dt, device="cuda")
    b = torch.empty(n, dtype=dt, device="cuda")
    p, q = C.c_void_p(At.data_ptr()), C.c_void_p(b.data_ptr())
    for _ in range(2):
        At.fill_(NAN)
        b.fill_(NAN)
        torch.cuda.synchronize()
        if harmonic:
            check(lib().mfb_assemble_harela(s._h, OMEGA, LAM_C.real, LAM_C.imag, MU_C.real, MU_C.imag,
                                            2000.0, 0.3, p, n + pad, q, None), "assemble")
        else:
            check(lib().mfb_assemble_staela(s._h, MU, 0.3, p, n + pad, q, None), "assemble")
    return At[:, :n].T.cpu().numpy(), b.cpu().numpy(), At[:, n:]


@pytest.mark.parametrize("pad", [0, 5])
@pytest.mark.parametrize("harmonic", [False, True])
@pytest.mark.parametrize("kind", KINDS)
def test_every_entry_is_stored(oracle, kind, harmonic, pad):
    import torch
    from multifebe_amd import bem
    bem._torch()
    m = _mesh(kind)
    A, b, between = _assemble(bem.BemSystem(m), harmonic, pad)
    kw = dict(lam_c=LAM_C, mu_c=MU_C, rho=2000.0, omega=OMEGA) if harmonic else dict(mu=MU, nu=0.3)
    Ao, bo = oracle.assemble(m, **{**kw, "nu": 0.3})
    n = m.n_dof - 3 * ("unused" in kind)
    assert np.all(np.abs(A - Ao)[:n] <= 1e-10 * np.abs(Ao[:n]).max(axis=1, keepdims=True))
    assert np.abs(b - bo)[:n].max() <= 1e-10 * np.abs(bo).max()
    assert torch.isnan(between).all()      # what lies between the columns is the caller's
    if "unused" in kind:
        assert not A[:, n:].any()
        x = np.random.default_rng(4).standard_normal((m.nn, 3)) * np.where(m.ctype == 0, 1e6, 1e-3)
        u, t = np.where(m.ctype == 0, m.cval, x), np.where(m.ctype == 0, x, m.cval)
        v = oracle.internal_points(m, m.x[-1:], u, t, **kw)[0]
        r = A[n:] @ x.ravel() - b[n:]
        assert np.abs(r + v).max() <= 1e-10 * np.abs(A[n:] * x.ravel()).max()


@pytest.mark.parametrize("harmonic", [False, True])
def test_collapsed_element(harmonic):
    from multifebe_amd import bem
    bem._torch()
    c, split, to = _collapsed()
    A, b, _ = _assemble(bem.BemSystem(c), harmonic)
    As, bs, _ = _assemble(bem.BemSystem(split), harmonic)
    P = np.zeros((split.n_dof, c.n_dof))
    P[np.arange(split.n_dof), (3 * to[:, None] + np.arange(3)).ravel()] = 1.0
    own = (3 * c.conn[0][:, None] + np.arange(3)).ravel()
    r = np.setdiff1d(np.arange(c.n_dof), own)
    rs = np.nonzero(P[:, r].any(axis=1))[0]      # their rows in the split boundary: one each
    ref, bref = As[rs] @ P, bs[rs]
    assert np.isfinite(A[r]).all() and np.isfinite(b[r]).all()
    assert np.abs(A[r] - ref).max() <= 1e-12 * np.abs(ref).max()
    assert np.abs(b[r] - bref).max() <= 1e-12 * np.abs(bref).max()


@pytest.mark.parametrize("kind", ["closed", "open", "unused open"])
def test_learned_rules(kind):
    import torch
    from multifebe_amd import bem
    from multifebe_amd.qnet import QNet
    m = _mesh(kind)
    net = QNet(0)
    with np.load(os.path.join(ROOT, "multifebe_amd", "data", "qnet_tau1e-10.npz")) as z:
        net.params = z["params"]
    out = []
    for learned in (False, True):
        s = bem.BemSystem(m, bem.Settings(qsi_relative_error=1e-8))
        if learned:
            s.set_qnet(net, 0.99, 1e-12, 0)
        At, b = s.alloc(True)
        At.fill_(NAN)
        b.fill_(NAN)
        out.append(s.assemble_harela(900.0, LAM_C, MU_C, 2000.0, 0.3, At, b))
    (A0, b0), (A1, b1) = out
    # the rules differ, each within its tolerance of 1e-8 of a pair's block; 1e-5 of the matrix is far above
    assert (A1 - A0).abs().max() <= 1e-5 * A0.abs().max()
    assert (b1 - b0).abs().max() <= 1e-5 * b0.abs().max()


def test_captured_batch_of_open_surfaces():
    """surfaces of different sizes whose extra rows share one buffer, static and harmonic"""
    import torch
    from multifebe_amd import bem
    bem._torch()
    jobs = []
    for k, kind in enumerate(["open", "unused open", "closed", "collapsed", "open"]):
        m = _collapsed()[0] if kind == "collapsed" else _mesh(kind)
        nodes = np.setdiff1d(np.arange(m.nn), m.conn[0]) if kind == "collapsed" else np.arange(m.nn)
        s = bem.BemSystem(m)
        for harmonic in (True, False):
            At, b = s.alloc(harmonic)
            j = dict(system=s, At=At, b=b, nu=0.3)
            j.update(dict(omega=700.0 + 200.0 * k, lam=LAM_C, mu_c=MU_C, rho=2000.0) if harmonic
                     else dict(mu=MU * (1 + k)))
            jobs.append((j, nodes))
    ref = []
    for j, nodes in jobs:
        s = j["system"]
        At, b = (s.assemble_harela(j["omega"], j["lam"], j["mu_c"], j["rho"], 0.3) if "omega" in j
                 else s.assemble_staela(j["mu"], 0.3))
        ref.append((At.T.cpu().numpy(), b.cpu().numpy()))
    g = bem.BatchGraph([j for j, _ in jobs])
    for replay in range(4):
        if replay == 3:
            for j, _ in jobs:
                j["At"].fill_(NAN)
                j["b"].fill_(NAN)
            bem.assemble_batch([j for j, _ in jobs])
        else:
            for j, _ in jobs:
                j["At"].fill_(NAN)
                j["b"].fill_(NAN)
            torch.cuda.synchronize()
            g.launch()
            g.check()
        for (j, nodes), (A, b) in zip(jobs, ref):
            r = (3 * nodes[:, None] + np.arange(3)).ravel()
            # the same sums, a few of them in another order
            d = np.abs(j["At"].T.cpu().numpy()[r] - A[r]).max()
            assert d <= 1e-13 * np.abs(A[r]).max(), (replay, d)
            assert np.abs(j["b"].cpu().numpy()[r] - b[r]).max() <= 1e-13 * np.abs(b[r]).max()
