"""FP32 panels of the LU choose LAPACK's pivots, with interchanges in nearly every column and with ties.

The FP32 matrices are P L U with known factors: L unit lower with entries of 0.5 / sqrt(n) at most, U
dominant on its diagonal, so that no rounding can change a pivot, P random.  In a tied column the
largest entry occurs in two rows, of one wave, of two or of two workgroups, and there is nothing else in
those rows of L nor in U's row and column, so that the two stay equal through the elimination: the first
of them is LAPACK's pivot, and the other one takes its place.
Columns are scaled by powers of two before they are rounded to FP32, which changes no pivot.
Factors: n eps_32 of the largest entry, and the factor 2 of |L| |U| over |A|.  The refinement gains four
digits a step at a condition below 10: five steps at most."""
import numpy as np
import pytest
import scipy.linalg as sla

pytestmark = pytest.mark.gpu

TIES = (0, 5, 31, 32, 33, 63, 64, 200, 300, 500, 511, 512, 1000, 1100, 1200)


def plu(n, cplx, ties):
    rng = np.random.default_rng(n + cplx)

    def rand(*s):
        a = rng.uniform(-1, 1, s)
        return 0.5 * (a + 1j * rng.uniform(-1, 1, s)) if cplx else a
    L = np.tril(rand(n, n), -1) * (0.5 / np.sqrt(n)) + np.eye(n)
    U = np.triu(rand(n, n), 1) / np.sqrt(n) + np.diag(1.0 + rng.random(n)) * (1j if cplx else 1.0)
    taken = set(ties)
    for k, j in enumerate(ties):
        U[j, j + 1:] = 0.0
        U[:j, j] = 0.0
        r = j + (1, 70, 300)[k % 3]
        while r in taken:
            r += 1
        if r < n:
            taken.add(r)
            L[r, :r] = 0.0
            L[r, j] = (-1.0, 1.0, 1j if cplx else -1.0)[k // 3 % 3]
    A = (L @ U)[rng.permutation(n)]
    # entries of 24 bits; a tied column's are one value up to sign and i
    return A.astype(np.complex64 if cplx else np.float32).astype(A.dtype)


@pytest.mark.parametrize("cplx", [False, True])
@pytest.mark.parametrize("n", [77, 512, 513, 1535, 1536, 1537])
def test_fp32_pivots_match_lapack(n, cplx):
    import torch
    from multifebe_amd import bem
    bem._torch()
    A = plu(n, cplx, [j for j in TIES if j < n - 3])
    lu, piv = sla.lu_factor(A)
    assert np.mean(piv != np.arange(n)) > 0.8
    b = np.asfortranarray(A @ np.ones((n, 1)))
    F, ipiv, z = np.asfortranarray(A), np.zeros(n, np.int32), np.zeros(n)
    solve = bem.solve_lse_c if cplx else bem.solve_lse_r
    rep = solve(n, F, ipiv, 0, None, b"N", z, z, 1, b, precision_mode=bem.PREC_FP32_REFINE)
    assert rep["precision_mode"] == bem.PREC_FP32_REFINE and rep["fell_back"] == 0
    assert np.array_equal(ipiv, piv + 1)
    assert np.abs(F - lu).max() <= 2 * n * 6e-8 * np.abs(lu).max()
    assert np.abs(b - 1.0).max() <= 1e-12 and rep["refinement_steps"] <= 5
    # the device entry point factorises the same way
    At = torch.from_numpy(np.ascontiguousarray(A.T)).cuda()
    x, rep = bem.gesv_device(At, torch.from_numpy(A @ np.ones(n)).cuda(), bem.PREC_FP32_REFINE)
    assert rep["fell_back"] == 0 and rep["refinement_steps"] <= 5
    assert (x - 1.0).abs().max().item() <= 1e-12
