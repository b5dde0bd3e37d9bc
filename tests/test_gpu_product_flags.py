"""The FP64 tangent's product with the flags and families that its kernels branch on:
discontinuity capturing, each tau, and a family of 64 rows or more above 32768 nodes, where
the slaves' sums are formed by lanes of their own.

Reference: the assembled tangent applied by SparseAp to the direction at the periodic
masters, folded by bc3per.  Bar, norm of the difference over the norm, each component scaled
by its largest value: 7.1e-14 (64 units of rounding, 2^-53, of a row's terms and a factor of
ten for rows that cancel) with a diagonal tau; the matrix tau is formed again from the
state by an eigenvalue decomposition whose condition takes further digits, 1e-12.  A family's
row adds up to 71 rows: a factor of ten, the square root of their number rounded up.
"""
import numpy as np
import pytest

from phasta_amd import config, mesh, solver

pytestmark = pytest.mark.gpu


def rel(a, b):
    return np.linalg.norm(a - b) / np.linalg.norm(b)


def check(case, params, tol):
    rng = np.random.default_rng(case.N)
    y = np.asfortranarray(case.yold[case.iper - 1])
    p = np.asfortranarray(rng.standard_normal((case.nshg, 5)))
    g = solver.GpuSolver(case, params=params)
    try:
        _, _, _, lhsk = g.elmgmrs(y, np.zeros_like(y))
        want = g.bc3per(g.sparse_ap(lhsk, np.asfortranarray(p[case.iper - 1])))
        got = g.tangent_ap(y, p)
    finally:
        g.close()
    scale = np.abs(want).max(axis=0)
    e = rel(got / scale, want / scale)
    print(f"[product] N={case.N} {e:.1e}", flush=True)
    assert e < tol


@pytest.mark.parametrize("N", [5, 33])
@pytest.mark.parametrize("idc,itau", [(0, 1), (1, 0), (2, 1), (0, 10), (1, 10)])
def test_product_with_flags(N, idc, itau):
    case = mesh.box_case(N, mach=0.3, kspace=2)
    check(case, config.solver_params(N, 0.3, 2, idc=idc, itau=itau),
          1e-12 if itau == 10 else 7.1e-14)


@pytest.mark.parametrize("slaves", [3, 63, 64, 70])
@pytest.mark.parametrize("N", [6, 33])
def test_product_with_a_large_family(N, slaves):
    case = mesh.box_case(N, mach=0.3, kspace=2)
    own = np.arange(1, case.nshg + 1)
    free = np.flatnonzero((case.iBC == 0) & (case.iper == own))
    free = free[~np.isin(free + 1, case.iper[case.iper != own])]
    case.iper[free[1:1 + slaves]] = free[0] + 1
    case.iBC[free[1:1 + slaves]] |= 1024
    check(case, None, 7.1e-13)
