"""The Krylov iteration's kernels at the sizes where they branch: every width
of the Gram-Schmidt kernel (1 to 60 basis vectors), vectors of odd and even
length, one and several workgroups, and periodic families inside and beyond a
64-row group.

Bar: the GPU runs the oracle's recurrence with its inner products taken in
one pass, so a K-step update differs by rounding amplified by the small
systems' conditioning: 1e-10 relative (60 steps x 1e-16 x a condition number
of 1e3 to 1e4 at most).
"""
import numpy as np
import pytest

import pyoracle
from phasta_amd import mesh, solver

pytestmark = pytest.mark.gpu
TOL = 1e-10


def rel(a, b):
    return np.linalg.norm(a - b) / np.linalg.norm(b)


# etol 0 runs exactly K iterations; 1e-10 ends the cycle by convergence
@pytest.mark.parametrize("N,K,etol", [(2, 1, 0.0), (4, 4, 0.0), (4, 5, 0.0), (5, 9, 0.0),
                                      (5, 13, 0.0), (7, 21, 0.0), (12, 33, 0.0), (12, 60, 0.0),
                                      (6, 60, 1e-10)])
def test_gmres_widths_against_oracle(N, K, etol):
    case = mesh.box_case(N, mach=0.3, kspace=K, etol=etol)
    print(f"[krylov] N={N} K={K} etol={etol} n={5 * case.nshg}", flush=True)
    orc = pyoracle.Oracle(case)
    y, ac = orc.itr_predict_bc(case.yold)
    ref = orc.solgmrs(y, ac)
    gpu = solver.GpuSolver(case)
    try:
        gpu.diagnostics(orth=True)
        out = gpu.solgmrs(y, ac)
    finally:
        gpu.close()
    print(f"[krylov] iKs {out['iKs']}/{ref['iKs']} Dy {rel(out['Dy'], ref['Dy']):.1e} "
          f"orth {out['orth_loss']:.1e}", flush=True)
    assert out["iKs"] == ref["iKs"]
    assert rel(out["Dy"], ref["Dy"]) < TOL
    assert abs(out["echeck"] - ref["echeck"]) <= 1e-8 * ref["unorm0"]
    assert out["orth_loss"] < K * np.finfo(float).eps * ref["unorm0"] / ref["echeck"]


@pytest.mark.parametrize("slaves", [3, 63, 64, 70])
def test_periodic_families_in_the_matvec(slaves):
    """One master with many slaves: a family of up to 64 rows is folded by
    the matvec in its row group, a larger one by the separate fold."""
    case = mesh.box_case(6, mach=0.3, kspace=3, etol=0.0)
    free = np.flatnonzero((case.iBC == 0) & (case.iper == np.arange(1, case.nshg + 1)))
    free = free[~np.isin(free + 1, case.iper[case.iper != np.arange(1, case.nshg + 1)])]
    assert len(free) > slaves
    m = free[0]
    case.iper[free[1:1 + slaves]] = m + 1
    case.iBC[free[1:1 + slaves]] |= 1024
    orc = pyoracle.Oracle(case)
    y, ac = orc.itr_predict_bc(case.yold)
    ref = orc.solgmrs(y, ac)
    gpu = solver.GpuSolver(case)
    try:
        out = gpu.solgmrs(y, ac)
    finally:
        gpu.close()
    print(f"[krylov] {slaves} slaves: Dy {rel(out['Dy'], ref['Dy']):.1e}", flush=True)
    assert out["iKs"] == ref["iKs"] == 3
    assert rel(out["Dy"], ref["Dy"]) < TOL
