"""Panels that one workgroup factorises and the ones several share: sizes on both sides of the lines.

A narrow block of the LU is one workgroup's when it has at most 512 rows (one row a thread) or 1536
(three rows a thread, types of up to 8 bytes); the pivots and factors are LAPACK's on either side,
where a column's largest entry occurs more than once (the first of them), and with an exactly
singular column.
"""
import numpy as np
import pytest
import scipy.linalg as sla

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def bem():
    import torch
    from multifebe_amd import bem as B
    assert torch.cuda.is_available()
    return B


def matrix(n, cplx, seed):
    rng = np.random.default_rng(seed)
    A = rng.standard_normal((n, n))
    return A + 1j * rng.standard_normal((n, n)) if cplx else A


def column_major(M):
    import torch
    return torch.from_numpy(np.ascontiguousarray(M.T)).cuda()


@pytest.mark.parametrize("cplx", [False, True])
@pytest.mark.parametrize("n", [5, 511, 512, 513, 1535, 1537, 1568])
def test_pivots_and_factors_match_lapack(bem, n, cplx):
    import torch
    A = matrix(n, cplx, n)
    ties = [r for r in (3, 4, 64, 510, 1534) if r < n]
    A[ties, 0] = 9.0   # the first column's largest entry, several times, in different waves
    b = matrix(n, cplx, n + 1)[:, 0]
    At, bt = column_major(A), torch.from_numpy(b.copy()).cuda()
    ipiv = torch.zeros(n, dtype=torch.int32, device="cuda")
    bem.gesv_device(At, bt, bem.PREC_FP64, ipiv=ipiv)
    lu, piv = sla.lu_factor(A)
    assert ipiv[0].item() == 4
    assert np.array_equal(ipiv.cpu().numpy(), piv + 1)
    # n eps and a growth of some hundreds: 1568 * 2.2e-16 * 300 = 1e-10
    assert np.max(np.abs(At.T.cpu().numpy() - lu)) <= 1e-10 * np.max(np.abs(lu))


@pytest.mark.parametrize("cplx", [False, True])
@pytest.mark.parametrize("n", [512, 1536, 1537])
def test_fp32_panels_refine_to_fp64(bem, n, cplx):
    import torch
    A = matrix(n, cplx, n) + 3.0 * np.sqrt(n) * np.eye(n)
    b = matrix(n, cplx, n + 1)[:, 0]
    x, rep = bem.gesv_device(column_major(A), torch.from_numpy(b.copy()).cuda(),
                             bem.PREC_FP32_REFINE)
    xr = np.linalg.solve(A, b)
    assert rep["precision_mode"] == bem.PREC_FP32_REFINE and rep["fell_back"] == 0
    # backward stable to n eps, condition below 10
    assert np.linalg.norm(x.cpu().numpy() - xr) <= 1e-11 * np.linalg.norm(xr)


@pytest.mark.parametrize("n", [512, 1537])
def test_zero_column_is_reported(bem, n):
    import torch
    A = matrix(n, False, n)
    A[:, n - 2] = 0.0
    with pytest.raises(Exception, match="singular"):
        bem.gesv_device(column_major(A), torch.ones(n, dtype=torch.float64, device="cuda"),
                        bem.PREC_FP64)
