"""Factors psi, chi, TT1..TT3 of the harmonic fundamental solution (bem_harela3d.f90:660-682): the code
that the kernels run, compiled for the host, against 50 digits over |kappa r| = 1e-3 .. 120.

Bars, relative to the larger of psi, chi and to the largest of TT1..TT3.  Below |kappa_2 r| = 1 a factor
is s^2 (lead + u) with |u| below lead: at most seven roundings of 1.1e-16 in it, 8e-16.  From 1 to 3
terms of 30 / |z|^2 (closed form) or of |z|^4 g (series) meet, 45 roundings: 5e-15.  Above, the phase
carries |kappa r| eps: 5e-15 + |kappa r| eps."""
import os
import subprocess

import numpy as np
import pytest

mp = pytest.importorskip("mpmath")
from multifebe_amd import build, mesh as M

SOURCE = r"""
#include <hip/hip_runtime.h>
#include <cstdio>
#include "mfbem_device.h"
#include "mfbem_types.h"
int main() {
  double v[7];
  while (scanf("%la %la %la %la %la %la %la", v, v + 1, v + 2, v + 3, v + 4, v + 5, v + 6) == 7) {
    mfb::HarParams p;
    mfb::host_har_params(v[0], v[1], v[2], v[3], v[4], v[5], &p);
    mfb::zd f[10];   // all factors at once, then t*'s and u*'s by themselves
    mfb::har_factors<true, true>(&p, v[6], 1.0 / v[6], true, f[0], f[1], f[2], f[3], f[4]);
    mfb::har_factors<false, true>(&p, v[6], 1.0 / v[6], true, f[5], f[6], f[7], f[8], f[9]);
    mfb::har_factors<true, false>(&p, v[6], 1.0 / v[6], true, f[5], f[6], f[7], f[8], f[9]);
    for (int k = 0; k < 10; k++) printf("%a %a ", f[k].re, f[k].im);
    puts("");
  }
}
"""


@pytest.fixture(scope="module")
def factors(tmp_path_factory):
    d = tmp_path_factory.mktemp("factors")
    (d / "f.hip").write_text(SOURCE)
    exe = str(d / "f")
    subprocess.run([build.HIPCC, "--offload-host-only", "-O1", "-std=c++17", "-I" + build.CSRC,
                    "-I" + os.path.join(build.ROOT, "include"), str(d / "f.hip"),
                    os.path.join(build.CSRC, "mfbem_tables.cpp"), "-o", exe, "-lquadmath"],
                   check=True, capture_output=True)

    def run(rows):
        text = "\n".join(" ".join(float(v).hex() for v in r) for r in rows) + "\n"
        out = subprocess.run([exe], input=text, capture_output=True, text=True, check=True).stdout
        v = np.array([[float.fromhex(w) for w in l.split()] for l in out.splitlines()])
        return v[:, 0::2] + 1j * v[:, 1::2]
    return run


def exact(lam_re, lam_im, mu_re, mu_im, rho, omega, r):
    lam, mu, r = mp.mpc(lam_re, lam_im), mp.mpc(mu_re, mu_im), mp.mpf(r)
    k1 = 1j * mp.mpf(omega) / mp.sqrt((lam + 2 * mu) / mp.mpf(rho))
    k2 = 1j * mp.mpf(omega) / mp.sqrt(mu / mp.mpf(rho))
    q, s = mu / (lam + 2 * mu), 1 / r
    w1, w2 = s * mp.exp(-k1 * r), s * mp.exp(-k2 * r)
    D = w2 * (s / k2 + (s / k2) ** 2) - w1 * (q * s / k1 + (s / k2) ** 2)
    return [w2 + D, w2 - q * w1 + 3 * D,
            2 * (k2 * w2 - q * k1 * w1) + 12 * s * (w2 - q * w1) + 30 * D * s,
            2 * q * w1 * s - 3 * w2 * s - k2 * w2 - 6 * D * s,
            (2 * q - 1) * k1 * w1 + (4 * q - 1) * w1 * s - 2 * w2 * s - 6 * D * s]


@pytest.mark.parametrize("lo,hi,bar", [(1e-3, 0.1, 8e-16), (0.1, 0.5, 8e-16), (0.5, 1.0, 8e-16),
                                       (1.0, 1.5, 5e-15), (1.5, 2.0, 5e-15), (2.0, 3.0, 5e-15),
                                       (3.0, 10.0, None), (10.0, 120.0, None)])
def test_factors(factors, lo, hi, bar):
    rng = np.random.default_rng(7)
    rows, kr = [], []
    for nu in (0.05, 0.2, 0.3, 0.4, 0.49):
        for xi in (0.0, 0.02, 0.1):
            _, mu, lam = M.elastic_constants(1e9, nu, xi)
            k = np.exp(rng.uniform(np.log(lo), np.log(hi), 60))
            for v, r in zip(k, rng.uniform(0.1, 3.0, k.size)):
                rows.append((lam.real, lam.imag, mu.real, mu.imag, 2000.0,
                             v * abs((mu / 2000.0) ** 0.5) / r, r))
                kr.append(v)
    got = factors(rows)
    with mp.workdps(50):
        for q, row in enumerate(rows):
            ex = exact(*row) * 2
            for part in (slice(0, 2), slice(2, 5), slice(5, 7), slice(7, 10)):
                scale = max(abs(v) for v in ex[part])
                err = max(float(abs(mp.mpc(complex(g)) - v) / scale)
                          for g, v in zip(got[q, part], ex[part]))
                assert err <= (bar if bar else 5e-15 + kr[q] * 2.2e-16), (row, kr[q], err)
