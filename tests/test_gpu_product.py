"""The FP64 tangent's product and the mixed path's refinement where their nodal
kernels differ: periodic slaves summed in their master's lane and apart (from
32768 nodes on), one wavefront and many workgroups, constrained rows.

The reference of the product is the assembled tangent applied by SparseAp to the
direction at the periodic masters, folded by bc3per.  Bar: both round a row's sum of at most 27 blocks of five products,
each an element sum, in another order: 64 units of rounding of the row's
largest terms, 64 x 2^-53 = 7.1e-15 of the product's norm when nothing
cancels; the random direction makes terms and sum of one size, and a factor of
10 is left for the rows where they are not.
"""
import numpy as np
import pytest

import pyoracle
from phasta_amd import mesh, solver

pytestmark = pytest.mark.gpu


def rel(a, b):
    return np.linalg.norm(a - b) / np.linalg.norm(b)


@pytest.mark.parametrize("N", [2, 5, 12, 33])
def test_product_against_assembled_tangent(N):
    case = mesh.box_case(N, mach=0.3, kspace=5, grade=1.0 if N % 2 else 1.1, cfl=3.0)
    rng = np.random.default_rng(N)
    y = np.asfortranarray(case.yold)
    p = np.asfortranarray(rng.standard_normal((case.nshg, 5)))
    ac = np.zeros_like(y)
    g = solver.GpuSolver(case)
    _, _, _, lhsk = g.elmgmrs(y, ac)
    want = g.bc3per(g.sparse_ap(lhsk, np.asfortranarray(p[case.iper - 1])))
    got = g.tangent_ap(y, p)
    g.close()
    scale = np.abs(want).max(axis=0)
    assert rel(got / scale, want / scale) < 7.1e-14


@pytest.mark.parametrize("N", [3, 33])
def test_refinement_reaches_the_fp64_solution(N):
    case = mesh.box_case(N, mach=0.3, kspace=20, grade=1.0, etol=1e-6)
    y, ac = np.asfortranarray(case.yold), np.zeros((case.nshg, 5), order="F")
    o = pyoracle.Oracle(case)
    y, ac = o.itr_predict_bc(case.yold)
    out = {}
    for prec in (solver.PHG_FP64, solver.PHG_MIXED):
        g = solver.GpuSolver(case, precision=prec)
        out[prec] = g.solgmrs(y, ac)
        g.close()
    a, b = out[solver.PHG_MIXED], out[solver.PHG_FP64]
    # both residuals are below etol: the updates differ by etol times the
    # scaled system's condition number, some 1e2 at this time step
    assert a["converged"] and a["echeck"] <= a["epsnrm"]
    assert rel(a["Dy"], b["Dy"]) < 1e-4
