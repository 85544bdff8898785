"""Narrow LU blocks: the persistent panels (one workgroup's and shared ones) and the path with a launch
per column, which an expired wait falls back to, give the same factors, bit by bit."""
import os
import subprocess
import sys

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

CHILD = """
import sys, numpy as np, torch
from multifebe_amd import bem
out = {}
for cplx in (0, 1):
    rng = np.random.default_rng(5)
    n = 700
    A = rng.standard_normal((n, n))
    if cplx:
        A = A + 1j * rng.standard_normal((n, n))
    At = torch.from_numpy(np.ascontiguousarray(A.T)).cuda()
    ipiv = torch.zeros(n, dtype=torch.int32, device="cuda")
    bem.gesv_device(At, torch.ones(n, dtype=At.dtype, device="cuda"), bem.PREC_FP64, ipiv=ipiv)
    out[f"lu{cplx}"], out[f"p{cplx}"] = At.cpu().numpy(), ipiv.cpu().numpy()
np.savez(sys.argv[1], **out)
"""


def test_column_path_gives_the_panels_bits(tmp_path):
    res = []
    for k, env in enumerate(({"MFB_LOOKAHEAD": "0"}, {"MFB_PANEL": "column"})):
        f = str(tmp_path / f"{k}.npz")
        subprocess.run([sys.executable, "-c", CHILD, f], env=dict(os.environ, **env), cwd=ROOT,
                       check=True, timeout=110)
        with np.load(f) as z:
            res.append({q: z[q] for q in z.files})
    for q in res[0]:
        assert np.array_equal(res[0][q], res[1][q]), q
